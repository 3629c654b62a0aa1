"""CPU: the split counts of Hessians of several planes fit the launch they make.

A product over several pairs of planes launches one workgroup per tile, pair and
split.  From the workspace that a Gram asks for (a 256x256 fp32 tile per
workgroup) the count per pair is read back.  `per_plane` is the count that fits
one launch per column plane best: the one taken is no lower (chains no longer),
and takes no more tokens, in full rounds of 256 workgroups of which each partial
tile counts as four, than that or one more, but for a 64th (where shorter chains
are as good as free they are taken).
"""
import pytest

from g2ptq_amd import _lib

PAIRS = {(0, 2): (9, 5), (1, 1): (4, 8), (2, 2): (6, 8)}  # pairs, most splits


def _cost(tiles, pairs, K, s):
    tokens = -(-K // (128 * s)) * 128
    groups = tiles * pairs * s
    return -(-groups // 256) * tokens + 4 * groups


@pytest.mark.parametrize("kind,dtype,C,K,per_plane", [
    (0, 2, 700, 1100, 1), (0, 2, 700, 2000, 1), (0, 2, 768, 4000, 2), (0, 2, 1280, 20000, 4),
    (0, 2, 2048, 8192, 4), (0, 2, 2752, 14000, 4), (0, 2, 4096, 16384, 3), (1, 1, 700, 2000, 1),
    (1, 1, 1000, 3000, 2), (1, 1, 2752, 14000, 8), (2, 2, 768, 4000, 2), (2, 2, 1000, 3000, 2),
    (2, 2, 2048, 8192, 7)])
def test_split_count_fits_all_pairs(kind, dtype, C, K, per_plane):
    pairs, most = PAIRS[kind, dtype]
    nt = -(-C // 256)
    tiles = nt * nt if kind == 1 else nt * (nt + 1) // 2  # GPTAQ's cross term asks for the most
    size = _lib.query_size("g2ptq_hessian_gram_ex_workspace", kind, dtype, K, C,
                           1 if kind == 2 else 0)
    s = size // (tiles * pairs * 256 * 256 * 4)
    assert size == tiles * pairs * s * 256 * 256 * 4
    assert per_plane <= s <= most
    for c in (per_plane, per_plane + 1):
        if c <= min(most, K // 512):
            assert _cost(tiles, pairs, K, s) <= _cost(tiles, pairs, K, c) * 65 // 64, (s, c)


def test_near_ties_take_shorter_chains():
    size = _lib.query_size("g2ptq_hessian_gram_ex_workspace", 0, 2, 14000, 2752, 0)
    assert size == 66 * 9 * 5 * 256 * 256 * 4  # 12 rounds of 2816 tokens for 10 of 3584


@pytest.mark.parametrize("kind,dtype,planes", [(0, 1, 2), (0, 2, 3), (1, 1, 2), (1, 2, 2), (2, 1, 2),
                                               (2, 2, 2)])
@pytest.mark.parametrize("C", [4096, 5120, 8192, 14336, 28672])
def test_workspaces_stay_within_what_staging_leaves_free(kind, dtype, planes, C):
    """Staging buffers leave 4 GiB of the device free: the partials of a Gram take no
    more than 3.5 of them, or than one launch per column plane takes."""
    for K in (4096, 16384, 204800):
        nt = -(-C // 256)
        tiles = nt * nt if kind == 1 else nt * (nt + 1) // 2
        size = _lib.query_size("g2ptq_hessian_gram_ex_workspace", kind, dtype, K, C,
                               1 if kind == 2 else 0)
        s = 1  # the largest power of two for 4096 workgroups of one column plane
        while s * 2 <= 16 // planes and tiles * planes * s < 4096:
            s *= 2
        assert size <= max(7 << 29, tiles * planes * s * 256 * 256 * 4), (K, size / 2 ** 30)
