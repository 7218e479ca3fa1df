"""Routing many tokens from features: the launch that takes several tokens per workgroup against the
one-token-per-workgroup launch of the same call in pieces. Priors, rings and statuses are the same
bytes (the dot products' order of summation is part of the interface)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PIECE = 200  # tokens of a call that stays with one token per workgroup


def _route(r, f, w, n, lo, hi):
    import torch

    rings = torch.zeros((hi - lo) * 40, dtype=torch.uint8, device="cuda")
    pri = torch.zeros((hi - lo, n), dtype=torch.float32, device="cuda")
    st = torch.full((hi - lo,), 7, dtype=torch.int32, device="cuda")
    r.route_features(f[lo:hi], w, rings, pri, st)
    torch.cuda.synchronize()
    return rings.cpu().numpy(), pri.cpu().numpy().view(np.uint32), st.cpu().numpy()


# 2, 4 and 8 tokens per workgroup with whole and ragged last workgroups; adapters at the edges of the
# 16, 32, 48 and 64 of a pass and above; feature counts below a chunk of 256, with and without a tail
@pytest.mark.parametrize("T,n,d", [(257, 16, 896), (385, 17, 260), (512, 33, 3584), (513, 48, 1000), (771, 64, 4),
                                   (1025, 5, 252), (1536, 1, 512), (1541, 65, 768), (2039, 64, 5120),
                                   (1600, 130, 1284), (1600, 600, 512), (4096, 32, 2048)])
def test_same_bytes_as_one_token_per_workgroup(hip, T, n, d):
    import torch

    rng = np.random.default_rng(T + n + d)
    f = rng.standard_normal((T, d), dtype=np.float32)
    f[T // 2, d // 2] = np.inf  # a token whose priors are not finite
    f[T - 1] = 0.0              # ties on every adapter
    w = rng.standard_normal((n, d), dtype=np.float32) * np.float32(0.05)
    ids = rng.permutation(n).astype(np.uint64)
    r = hip.Router(n, min(n, 8), 1.0, 0.02, 1.0, ids)
    if n > 4:
        r.set_policy_mask((rng.random(n) > 0.2).astype(np.uint8))
    fd, wd = torch.from_numpy(f).cuda(), torch.from_numpy(w).cuda()
    whole = _route(r, fd, wd, n, 0, T)
    assert whole[2][T // 2] == -1
    for lo in range(0, T, PIECE):
        hi = min(lo + PIECE, T)
        rings, pri, st = _route(r, fd, wd, n, lo, hi)
        assert np.array_equal(pri, whole[1][lo:hi]), f"priors of tokens {lo}..{hi}"
        assert np.array_equal(st, whole[2][lo:hi])
        a, b = (hip.rings_from_bytes(x).copy() for x in (rings, whole[0][40 * lo : 40 * hi]))
        ok = st == 0
        a["current_pos"][ok] += lo  # a ring holds its token's place in the call
        assert a.tobytes() == b.tobytes(), f"rings of tokens {lo}..{hi}"
