"""How many tokens a workgroup of a plain router call takes (CPU), and that a call at either side of the line
between one token and several gives the same bytes (GPU; the launches themselves: test_gpu_router_tokens)."""
import numpy as np
import pytest

import aoship

# (tokens, adapters, features) where one token each is the faster launch, and their neighbours past the line:
# more waves, shorter rows, or more workgroups than fit
FEW = [(257, 2, 3584), (600, 4, 3584), (1100, 2, 5120), (1664, 2, 3584), (1109, 3, 3584), (640, 4, 3200), (1792, 1, 5120),
       (426, 6, 4800)]
MANY = [(1665, 2, 3584), (1110, 3, 3584), (641, 4, 3200), (600, 4, 3196), (1793, 1, 5120), (427, 6, 4800), (384, 16, 5120),
        (257, 64, 896)]


@pytest.mark.parametrize("T,n,d", FEW + [(256, 64, 5120), (1, 16, 3584)])
def test_one_token_each(T, n, d):
    assert aoship.route_tokens(T, n, d) == 1


@pytest.mark.parametrize("T,n,d", MANY)
def test_several_tokens(T, n, d):
    tt = aoship.route_tokens(T, n, d)
    assert tt in (2, 4, 8) and (tt == 8 or T <= 256 * tt) and T > 128 * tt
    assert 4 * tt * n <= 16 * 1024


@pytest.mark.parametrize("T,n,d", [(20000, 600, 5120), (20000, 2000, 512), (20000, 4096, 512)])
def test_priors_fit_beside_the_stages(T, n, d):
    tt = aoship.route_tokens(T, n, d)
    assert tt == max(1, min(8, 1 << ((4096 // n).bit_length() - 1) if n <= 4096 else 1))


@pytest.mark.gpu
@pytest.mark.parametrize("T,n,d", FEW + MANY[:6])
def test_same_bytes_at_the_line(hip, T, n, d):
    from test_gpu_router_tokens import test_same_bytes_as_one_token_per_workgroup as same_bytes

    same_bytes(hip, T, n, d)
