"""Which way a step's short extends go (``Route``): the three ways at steps where
each was measured fastest, and the lists' capacities, which in an eager step are
the exact numbers of blocks."""
import pytest

from tokenfactory_amd import _native
from tokenfactory_amd.attention import Route

BF16, FP8 = _native.TF_DTYPE_BF16, _native.TF_DTYPE_FP8_E4M3
CUS = 256


def route(ext, max_len, fp8=False, exact=True, hq=24, hkv=4, d=256):
    n_work = sum(hkv * -(-e * (hq // hkv) // 256) for e in ext if e > 1)
    return Route(ext, sum(ext), hq, hkv, d, FP8 if fp8 else BF16, n_work, exact=exact,
                 max_len=max_len, cus=CUS)


@pytest.mark.parametrize("groups,ext,max_len,fp8", [
    # few requests, or long contexts of different lengths: units of 32 rows
    (2, [4] * 20, 8000, False), (2, [6] * 20, 8000, False), (2, [5] * 64, 8000, False),
    (2, [1] * 64 + [4] * 16, 8192, False), (2, [5] * 64, 8000, True),
    # units of 16 rows: rows that fit one, decodes beside few extends, fp8 decodes
    (1, [2] * 64, 8000, False), (1, [2] * 200, 300, False), (1, [1] * 64 + [3], 8192, False),
    (1, [1] * 100 + [3] * 8, 1000, False), (1, [1] * 8 + [4], 65536, True),
    (1, [1] * 48 + [4] * 16, 8192, True),
    # extend kernel: one entry per CU or more, two units each or short contexts
    (0, [10] * 64, 2010, False), (0, [8] * 256, 1500, False), (0, [10] * 400, 610, False),
    (0, [6] * 64, 8000, False), (0, [4] * 128, 300, False), (0, [10] * 64, 2010, True),
    (0, [1] * 900 + [4] * 200, 500, False),
])
def test_ways_of_short_extends(groups, ext, max_len, fp8):
    r = route(ext, max_len, fp8)
    assert r.row_groups == groups
    n_dec = ext.count(1)
    if groups:
        unit = 16 * groups
        assert r.n_blocks == sum(-(-e * 6 // unit) for e in ext)
        assert r.run_rows and not r.run_extend and r.n_pieces == 0 and not r.split
    else:
        assert r.n_blocks == 0 and r.run_extend and r.run_rows == (n_dec > 0)
        assert not r.split and not r.planned


def test_long_extends_keep_their_kernel():
    r = route([300, 4, 1, 1], 4000)
    assert r.row_groups and r.run_extend and r.run_rows
    assert r.n_blocks == 1 * (2 if r.row_groups == 1 else 1) + 2
    many = route([300] + [10] * 300 + [1], 3000)
    assert not many.row_groups and not many.split and many.run_extend and many.run_rows


@pytest.mark.parametrize("d,ext", [(128, [1, 70, 3, 1, 500]), (64, [33] * 5)])
def test_other_head_dims_count_exactly(d, ext):
    r = route(ext, 900, hq=32, hkv=8, d=d)
    assert r.row_groups == 2 and r.n_blocks == sum(-(-e * 4 // 32) for e in ext)
    assert r.n_blocks <= route(ext, 900, exact=False, hq=32, hkv=8, d=d).n_blocks


@pytest.mark.parametrize("ext,max_len", [([4] * 20, 8000), ([10] * 64, 2010), ([2] * 9 + [1], 700)])
def test_a_captured_step_has_room_for_any_lengths(ext, max_len):
    """Of the same T and B: every request of up to 64 rows in units of this height."""
    r = route(ext, max_len, exact=False)
    if r.row_groups:
        unit = 16 * r.row_groups
        assert r.n_blocks >= len(ext) * -(-64 // unit)
    assert r.run_extend and r.run_rows
