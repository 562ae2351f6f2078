"""The rule that cuts a padded prefill's keys into pieces (csrc/fa2_split_rule.h), on the CPU."""
import ctypes
import itertools

import pytest

from host_rules import rules

BODY = """
void plan(int64_t cus, int64_t B, int64_t Hq, int64_t Hkv, int64_t T, int64_t S, int64_t unit, int* out) {
  const mi_fa2::SplitPlan p = mi_fa2::split_plan(cus, B, Hq, Hkv, T, S, unit);
  out[0] = (int)p.tiles, out[1] = p.pieces, out[2] = p.each;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    fn = rules(tmp_path_factory.mktemp("rule"), "fa2_split_rule.h", BODY).plan
    fn.argtypes = [ctypes.c_int64] * 7 + [ctypes.c_int * 3]

    def ask(B, Hq, Hkv, T, S, unit=128, cus=256):
        out = (ctypes.c_int * 3)()
        fn(cus, B, Hq, Hkv, T, S, unit, out)
        return tuple(out)
    return ask


SHAPES = list(itertools.product((1, 3), ((12, 2), (1, 1), (17, 1)), (2, 40, 150, 700),
                                (100, 1000, 2048, 8192, 100000)))


def test_every_key_is_in_one_piece_and_no_piece_is_empty(plan):
    for (B, (Hq, Hkv), T, S), unit in itertools.product(SHAPES, (128, 256, 512, 2048, 4096)):
        tiles, pieces, each = plan(B, Hq, Hkv, T, S, unit)
        if pieces > 1:
            assert (pieces - 1) * each * unit < S <= pieces * each * unit
            assert tiles * pieces <= 256


def test_larger_units_fit_the_workspace_of_128_keys(plan):
    # the workspace query does not know the block size
    for (B, (Hq, Hkv), T, S), unit, cus in itertools.product(SHAPES, (256, 1024, 4096), (256, 64, 32)):
        assert plan(B, Hq, Hkv, T, S, unit, cus)[1] <= plan(B, Hq, Hkv, T, S)[1]
        assert plan(B, Hq, Hkv, T, S, 128, cus)[1] <= plan(B, Hq, Hkv, T, S)[1]


def test_blocks_that_leave_too_few_pieces_stay_whole(plan):
    """With few large blocks the pieces' chains are hardly shorter than the whole."""
    assert plan(1, 12, 2, 150, 2048)[1] > 1
    for T, S, block in ((5, 2048, 2048), (150, 2048, 2048), (400, 4000, 4096), (150, 2100, 2048)):
        assert plan(1, 12, 2, T, S, block)[1] == 1
    assert plan(1, 12, 2, 150, 8192, 2048)[1:] == (4, 1)
