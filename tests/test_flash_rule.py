"""Which steps the flash attention of paired waves takes (csrc/attention.hip, pair_form): a rule on counts, with 256 CUs where no device is
there to ask."""
import random

import pytest

from dinfer_amd.kernels import ops


def form(new, H, Hkv, page=16, longest=None):
    return ops.attn_flash_form(sum(new), len(new), longest or max(new), H, Hkv, page)


@pytest.mark.parametrize("H,Hkv,new", [
    # few rows of many kv heads: a tile of 256 columns is nearly empty
    (64, 64, [20] * 21), (64, 64, [531]), (32, 32, [60, 77, 8, 30, 44, 52, 70, 9, 12, 33, 71, 40, 28, 55, 61, 17, 22, 66, 35]),
    # one round of workgroups, or less: the longest of them is the time
    (16, 8, [134, 70, 95, 19, 40, 110, 128, 90, 77, 101, 83, 60, 25, 33, 130, 99, 47, 118, 65, 109, 88, 51]),
    (16, 4, [2, 588, 14, 23, 4, 275, 301, 2001]), (16, 8, [130] * 8), (40, 8, [1] * 31 + [512]), (16, 8, [1000, 1000]), (32, 8, [1000])])
def test_steps_that_were_slower_keep_the_tile_of_rows(H, Hkv, new):
    assert form(new, H, Hkv) == 0


@pytest.mark.parametrize("H,Hkv,new,want", [(32, 8, [2001], 2), (32, 8, [2500], 1), (32, 8, [4000], 1), (16, 8, [2600], 2), (32, 8, [500] * 4, 1),
                                            (32, 8, [256] * 16, 1), (40, 8, [100] * 16, 1), (32, 8, [1] * 30 + [4000], 1)])
def test_steps_that_gain_take_the_paired_waves(H, Hkv, new, want):
    assert form(new, H, Hkv) == want


def test_pages_that_the_paired_waves_cannot_read_and_odd_counts():
    for page in (8, 24, 40, 48):
        assert form([4000], 32, 8, page) == 0
    rng = random.Random(2)
    for _ in range(500):     # counts of a padded step: the longest is a bound
        new = [rng.randint(1, rng.choice((3, 300, 3000))) for _ in range(rng.randint(1, 70))]
        H, Hkv = rng.choice(((1, 1), (8, 1), (48, 8), (5, 5), (128, 8)))
        assert form(new, H, Hkv, longest=1 << (max(new) - 1).bit_length()) in ((0, 1, 2) if len(new) == 1 else (0, 1))
