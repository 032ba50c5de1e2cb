"""The width of a prefill launch (128 or 256 query rows per work group) against
measurements, and the rule's parts against their definitions (no GPU)."""

import heapq
import random

import numpy as np
import pytest
import torch

from mini_vllm.attention import paged_attention_gpu as pag

# (q heads, kv heads, head_dim), prefixes, chunks, us with 128 rows, with 256
MEASURED = [
    ((14, 2, 64), [0], [132 * 18], 27.0, 43.7),        # 264 units of 128 rows, one prompt
    ((14, 2, 64), [1536], [224 * 18], 75.0, 99.1),     # 448
    ((14, 2, 64), [1536], [256 * 18], 88.2, 111.2),    # 512
    ((8, 8, 64), [1536], [40 * 128], 67.9, 113.1),     # 320
    ((8, 8, 64), [0], [56 * 128], 74.1, 121.3),        # 448
    ((12, 3, 64), [0], [128 * 32], 50.6, 80.5),        # 384
    ((16, 1, 128), [0], [320 * 8], 43.4, 65.6),        # 320
    ((28, 4, 128), [0], [80 * 18], 29.9, 41.9),        # 320
    ((28, 4, 128), [1536] * 7, [504] * 7, 130.6, 108.0),  # 784: four rounds of 128, two of 256
    ((16, 1, 128), [0] * 9, [512] * 9, 32.7, 23.4),    # 576: three and two
    ((12, 3, 64), [0] * 11, [512] * 11, 20.2, 15.7),   # 528
    ((14, 2, 64), [0] * 14, [504] * 14, 26.5, 20.4),   # 784
    ((28, 4, 128), [0] * 32, [40] * 32, 15.8, 10.6),   # short chunks, 384
    ((28, 4, 128), [300] * 65, [17] * 65, 29.7, 24.5),  # one block each, 260
    ((14, 2, 64), [2000] * 130, [5] * 130, 43.1, 55.5),  # over long prefixes
    ((8, 8, 64), [2000] * 75, [17] * 75, 77.6, 98.5),   # 600
    ((28, 4, 128), [0] * 32, [17] * 32, 8.8, 7.3),     # one round, few keys
    ((28, 4, 128), [0], [456 * 18], 473.0, 434.0),     # over four rounds
    ((14, 2, 64), [1536] * 16, [512] * 16, 82.5, 75.4),  # 928
]


@pytest.mark.parametrize("heads,cached,qlens,narrow_us,wide_us", MEASURED)
def test_the_faster_width_is_taken(heads, cached, qlens, narrow_us, wide_us):
    narrow, wide = pag._prefill_block_tokens(*heads, torch.bfloat16)
    got = pag._prefill_tokens(*heads, torch.bfloat16, 256, cached, qlens)
    assert got == (narrow if narrow_us < wide_us else wide)


def test_one_round_keeps_128_rows():
    """Their two sets of waves share the keys, except over few keys."""
    for qlens in ([37], [512] * 4, [1] * 128):
        assert pag._prefill_tokens(14, 2, 64, torch.float16, 256, [1536] * len(qlens), qlens) == 18
    assert pag._prefill_tokens(14, 2, 64, torch.float32, 256, [0], [10 ** 5]) == 16  # one size
    assert pag._prefill_tokens(14, 2, 64, torch.bfloat16, 256, [5, 0], [0, 0]) == 18
    with pytest.raises(RuntimeError, match="not supported"):
        pag._prefill_tokens(17, 1, 64, torch.bfloat16, 256, [0], [5])


def test_short_launches_take_the_fewest_rows_of_one_round():
    """head_dim 128: 32, 64, 96 or 128 rows, as the CUs hold their groups; not
    at 64, and not where keys are cut into parts."""
    def tokens(heads, n, q, cached=0):
        return pag._prefill_tokens(*heads, torch.bfloat16, 256, [cached] * n, [q] * n)

    big = (28, 4, 128)  # 7 query heads per kv head: 4, 9, 13 and 18 tokens
    assert tokens(big, 1, 37) == 4 and tokens(big, 1, 256) == 4   # 64 blocks x 4 heads
    assert tokens(big, 1, 257) == 9 and tokens(big, 7, 75) == 9   # 7 x 9 x 4 = 252
    assert tokens(big, 16, 42) == 13 and tokens(big, 21, 42) == 18
    assert tokens((16, 1, 128), 1, 20) == 2 and tokens((6, 6, 128), 1, 200) == 32
    assert tokens(big, 1, 37, 731) == 4 and tokens(big, 1, 37, 732) == 18  # 768 keys
    assert tokens((14, 2, 64), 1, 37) == 18


def test_width_of_a_launch_with_lengths_on_the_device():
    def fixed(rows, seqs, d):
        return pag._prefill_tokens_fixed(14, 2, d, torch.bfloat16, 256, rows, seqs)

    for d in (64, 128):
        assert fixed(18 * 512, 1, d) == 18  # 1024 units: four rounds
        assert fixed(18 * 512 + 1, 1, d) == 36
    assert fixed(18 * 40, 40, 64) == 18 and fixed(18 * 40, 40, 128) == 36
    assert fixed(18 * 60 + 1, 60, 128) == 18
    # one round of fewer rows: (blocks + sequences) x 2 heads
    assert fixed(37, 1, 64) == 18 and fixed(37, 1, 128) == 4 and fixed(4 * 127, 1, 128) == 4
    assert fixed(4 * 127 + 1, 1, 128) == 9


def test_blocks_cover_every_token_once():
    rng = random.Random(3)
    for _ in range(50):
        n = rng.randint(1, 9)
        cached = np.array([rng.choice([0, rng.randint(0, 3000)]) for _ in range(n)])
        qlens = np.array([rng.choice([0, 1, rng.randint(0, 200)]) for _ in range(n)])
        t = rng.choice([1, 8, 18, 36, 128])
        got = sorted(zip(*(x.tolist() for x in pag._prefill_blocks(cached, qlens, t))))
        want = [(i, t0, min(t, q - t0), c + min(q, t0 + t))
                for i, (c, q) in enumerate(zip(cached.tolist(), qlens.tolist()))
                for t0 in range(0, q, t)]
        assert got == sorted(want)


def test_launch_time_is_a_bound_near_the_list_schedule():
    """Never above the time of the longest-first schedule of the groups over
    the CUs, and at most a group's time below it."""
    rng = random.Random(4)
    for _ in range(200):
        hkv, cus = rng.choice([1, 2, 3, 8]), rng.choice([4, 16, 256])
        cost = [rng.choice([1.0, rng.uniform(.2, 9)]) for _ in range(rng.randint(1, 60))]
        busy = [0.0] * cus
        for c in sorted(cost * hkv, reverse=True):
            heapq.heapreplace(busy, busy[0] + c)
        got = pag._prefill_us(np.array(cost), hkv, cus)
        assert got <= max(busy) + 1e-9
        assert max(busy) <= got + max(cost)
