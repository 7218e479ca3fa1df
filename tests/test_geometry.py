"""Decode launch geometry (CPU): every wave of every GEMV launch gets at least one K group.

The decode GEMVs split K over the waves of a workgroup and over ks workgroups per row block. Where
the waves read the activations themselves (3 or more tokens, in general) a wave with no group would
read before the row block; where the activations are staged, the LDS budget can force more splits
than the waves per workgroup allow, and the geometry then falls back to 4-wave workgroups. This
replays the library's own choice (the same function the forwards call) for every workload shape at
every decode token count, over narrow and wide adapter tables.
"""
import pytest

import aoship

# (hidden, intermediate) of the MLP shapes: the 0.5B plumbing layer, the 7B layer, the 32B
# stress layer; then projection row counts sharing one input (q+k+v, o) at their input widths.
MLP_SHAPES = [(896, 4864), (3584, 18944), (5120, 27648)]
LARGE_SHAPES = [(8192, 28672), (16384, 53248)]
PROJ_SHAPES = [(3072 + 1024 + 1024, 3072), (3072, 3072), (3584 + 512 + 512, 3584), (3584, 3584),
               (152064, 3584)]
# x-shrink rank rows (adapters x padded rank x modules) and h-shrink rows
SHRINK_ROWS = [(8 * 16 * 2, 896), (16 * 16 * 2, 3584), (32 * 16 * 3, 3072), (64 * 64 * 2, 5120),
               (16 * 48 * 2, 3584)]
H_SHRINK_ROWS = [(8 * 16, 4864), (16 * 16, 18944), (64 * 64, 27648), (16 * 48, 18944)]
# adapter tables: none, 16 of rank 16, 64 of rank 64
TABLES = [(0, 0), (16, 16), (64, 64)]
LAUNCHES = [(k, o, i) for H, I in MLP_SHAPES + LARGE_SHAPES for k, o, i in ((0, I, H), (1, H, I))] + [(2, o, i) for o, i in PROJ_SHAPES]
# few K groups: the fewest that a launch reading x itself takes (8), and fewer; few and many row blocks
LAUNCHES += [(k, o, 64 * G) for k in (0, 1, 2) for o in (32, 96, 4096) for G in (4, 5, 7, 8, 9, 15, 16, 17, 33)]


@pytest.mark.parametrize("T", range(1, 33))
@pytest.mark.parametrize("n,rpad", TABLES)
def test_every_gemv_wave_gets_a_group(T, n, rpad):
    for kind, out, inp in LAUNCHES:
        G = inp // 64
        direct, w, ks, wr, g = aoship.decode_launch(kind, out, inp, T, n=n, rpad=rpad)
        case = f"kind {kind} {out}x{inp} T={T} n={n}: direct {direct}, waves {w}, splits {ks}, rows {wr}"
        assert w in (4, 8) and 1 <= ks <= G and wr in (1, 2, 4, 8) and w % wr == 0, case
        assert wr == 1 or T > 2, "1-2 tokens keep one row block per workgroup (the h shrink needs it)"
        assert g >= 1, case
        groups = out // 32 * G  # large launches of few tokens stage x, and gate/up over a wide table
        staged = kind == 0 and (n * rpad > 1024 or 100000 < groups <= 200000)
        staged |= kind == 1 and min(n, 8 * T) * rpad <= 1280 and 60000 < groups <= 200000
        assert direct == (T > 2 and G >= 8 and not (staged and T <= 8)), case
        if direct:  # 4 waves on one row block, 1 to 48 K groups for each wave of its splits
            assert w == 4 and wr == 1 and 4 * ks <= G and (-(-G // (4 * ks)) <= 48 or groups > 200000), case
        else:
            budget = (64 if w == 8 and T > 2 else 32) * 1024
            assert 128 + T * -(-G // ks) * 136 <= budget, f"staged x exceeds the LDS budget: {case}"


# (kind, row blocks, K groups): 7B q/k/v, 32B o and down, gate/up of hidden 4096
@pytest.mark.parametrize("kind,rb,G", [(2, 144, 56), (2, 160, 80), (1, 160, 432), (0, 344, 64)])
@pytest.mark.parametrize("T", [3, 8, 9, 32])
def test_wide_unions_get_more_waves(kind, rb, G, T):
    """Over 64 adapters of rank 64 (up to 256 expand steps of each row block) a launch that reads x itself has
    at least half as many splits again; over the columns of the line and below, the narrow table's."""
    if kind == 0 and T <= 8:
        return  # staged
    narrow = aoship.decode_geometry(kind, 32 * rb, 64 * G, T, n=32, rpad=16)[1]
    line = aoship.decode_geometry(kind, 32 * rb, 64 * G, T, n=64 if T > 8 else 32, rpad=16)[1]
    wide = aoship.decode_geometry(kind, 32 * rb, 64 * G, T, n=64, rpad=64)[1]
    assert narrow == line and (2 * wide >= 3 * narrow or -(-G // (4 * wide)) <= 48), (narrow, line, wide)


# (kind, row blocks, K groups, tokens, adapters, rank, splits): more splits only where they were measured to pay
@pytest.mark.parametrize("kind,rb,G,T,n,r,ks", [
    (2, 128, 64, 8, 12, 64, 2), (2, 159, 64, 3, 24, 32, 2), (2, 160, 64, 8, 12, 64, 1), (2, 234, 26, 3, 19, 32, 1),
    (2, 322, 18, 7, 60, 16, 1), (2, 127, 64, 8, 12, 64, 2), (2, 128, 64, 8, 8, 64, 1), (2, 128, 64, 9, 12, 64, 1),
    (1, 112, 296, 16, 64, 64, 3), (1, 32, 147, 20, 49, 32, 8), (1, 160, 432, 16, 64, 64, 3), (1, 160, 432, 16, 16, 16, 3)])
def test_splits_of_launches_over_wide_tables(kind, rb, G, T, n, r, ks):
    direct, _, got, _, _ = aoship.decode_launch(kind, 32 * rb, 64 * G, T, n=n, rpad=r)
    assert direct and got == ks


@pytest.mark.parametrize("T", range(3, 33))
def test_every_wave_of_a_pinned_staged_launch_gets_a_group(T):
    """Pinned to any one row split, the launches stage x: 8 waves over a long K with up to 64 KB of it."""
    for kind, out, inp in LAUNCHES[: 2 * len(MLP_SHAPES + LARGE_SHAPES) + len(PROJ_SHAPES)]:
        for wr_pin in (1, 2, 4, 8):
            direct, w, ks, wr, g = aoship.decode_launch(kind, out, inp, T, wr_pin=wr_pin)
            case = f"kind {kind} {out}x{inp} T={T} pin {wr_pin}: waves {w}, splits {ks}, rows {wr}"
            assert not direct and w in (4, 8) and 1 <= ks <= inp // 64 and w % wr == 0 and g >= 1, case
            assert 128 + T * -(-(inp // 64) // ks) * 136 <= (64 if w == 8 else 32) * 1024, case


@pytest.mark.parametrize("T", range(1, 33))
def test_shrink_geometry_within_limits(T):
    """Shrinks: the K splits stay within the groups and the LDS budget (32 KB). A shrink wave may get no
    group when its launch runs more waves per workgroup than its splits leave groups; it then
    reads the zero row and adds nothing."""
    for kind, shapes in ((3, SHRINK_ROWS), (4, H_SHRINK_ROWS)):
        for rows, inp in shapes:
            w, ks, _, g = aoship.decode_geometry(kind, rows, inp, T)
            G = inp // 64
            assert 1 <= ks <= G
            assert 128 + T * -(-G // ks) * 128 <= 32 * 1024


@pytest.mark.parametrize("T", [1, 2])
@pytest.mark.parametrize("wr", [1, 2, 4])
@pytest.mark.parametrize("ks", [0, 1, 2, 4])
def test_pinned_gate_up_keeps_one_row_block_at_one_or_two_tokens(T, wr, ks):
    """A pinned row-split shape is not applied to the 1-2 token gate/up launch, whose wave 0 forms
    the h shrink's partials for the workgroup's one row block; other launches take the pin."""
    for H, I in MLP_SHAPES:
        w, k, r, g = aoship.decode_geometry(0, I, H, T, wr, ks)
        assert r == 1 and g >= 1
        if ks and (H // 64) // ks >= w:  # a pin that leaves a wave without a K group is not applied
            assert k == ks
    w, k, r, g = aoship.decode_geometry(0, 18944, 3584, 3, 4, 0)
    assert r == 4


def test_geometry_rejects_bad_shapes():
    with pytest.raises(aoship.AosError):
        aoship.decode_geometry(0, 3584, 100, 1)
    with pytest.raises(aoship.AosError):
        aoship.decode_geometry(0, 3584, 3584, 33)
    with pytest.raises(aoship.AosError):
        aoship.decode_geometry(0, 3584, 3584, 3, n=4, rpad=20)
