"""The plan's piece bound where few (sequence, kv head) units share the CUs.

Fewer units than half the CUs: pieces of at least sqrt(tiles / 2) tiles of the
longest sequence, down to a multiple of four (up where at most 1.5 are missing),
one group per CU up to 32 tiles per CU and 34 per CU that equal pieces of every
unit fill (192 of 256 for 96 units), else two. The bound both plan kernels pick must be the smallest one that fits
under these rules (brute force), and the decode on it must match the oracle.
"""

import math

import pytest
import torch

from benchmarks.paged_decode_workloads import WorkloadSpec, make_case
from gpu_util import DEV, TOL, oracle_step, say, to_device
from mini_vllm.attention import paged_attention_gpu as pag

pytestmark = pytest.mark.gpu


def _bound(kv_lens, hkv, per_cu, cus):
    tiles = [(k + 15) // 16 for k in kv_lens]
    units, total, most = len(tiles) * hkv, sum(tiles), max(tiles)
    few = 2 * units < cus
    one = few and total * hkv <= min(32 * cus, 34 * (cus // units * units))
    target = cus * (1 if one else min(2, per_cu))
    l_cap = 511
    l_min = min(l_cap, max(4, -(-most // 128), int(math.sqrt(most / 2) + 1.5) // 4 * 4 if few else 0))
    l_top = min(l_cap, max(l_min, most))
    l_fair = min(l_cap, max(l_min, -(-(total * hkv) // target)))

    def groups(l):
        return hkv * sum(-(-t // l) for t in tiles)

    if groups(l_top) > target:
        return l_fair
    l = min(l_fair, l_top)
    while groups(l) > target:
        l += 1
    return max(l_min, min(l_cap, 2 * l_fair)) if l > 2 * l_fair else l


@pytest.mark.parametrize("hq,hkv,d,dtype,lens", [
    (14, 2, 64, torch.bfloat16, [1]), (14, 2, 64, torch.bfloat16, [4096]),
    (14, 2, 64, torch.float32, [701]), (14, 2, 64, torch.float16, [512, 511, 513, 528]),
    (14, 2, 64, torch.bfloat16, [4096] * 16), (14, 2, 64, torch.bfloat16, [4112] * 16),
    (28, 4, 128, torch.bfloat16, [2048] * 8), (8, 8, 64, torch.float16, [300] * 15),
    (8, 8, 64, torch.float16, [300] * 16), (16, 1, 128, torch.float32, [30, 9000, 2]),
    (14, 2, 64, torch.bfloat16, [1000] * 48), (14, 2, 64, torch.bfloat16, [1300] * 48),
    (8, 8, 64, torch.float16, [1100] * 12), (12, 3, 64, torch.float16, [1300] * 32),
    (14, 2, 64, torch.bfloat16, [700] * 63), (14, 2, 64, torch.bfloat16, [700] * 64),
], ids=lambda v: str(v)[:24])
def test_bound_and_decode(hq, hkv, d, dtype, lens):
    say("plan, few units", hq, hkv, d, dtype, len(lens), max(lens))
    case = make_case(WorkloadSpec("few", hq, hkv, d, 16, dtype, len(lens), ("fixed", lens)), seed=51,
                     nan_fill=True)
    c = to_device(case)
    plan = pag.plan_decode(c.block_table, c.kv_len, 16, case.layout.num_blocks, DEV, d, dtype, hkv)
    per_cu, cus = pag._groups_per_cu(DEV, d, dtype)
    want = _bound(lens, hkv, per_cu, cus)
    assert plan.partition_tokens == 16 * want
    assert plan.num_groups == hkv * sum(-(-((k + 15) // 16) // want) for k in lens)
    pag.hip_cache_write(c.new_key, c.new_value, c.key_cache, c.value_cache, c.slot_mapping, 16)
    out = pag.hip_decode_attention(c.query, c.key_cache, c.value_cache, c.block_table, c.kv_len, 16)
    ref, _, _ = oracle_step(case)
    err = (out.float().cpu() - ref).abs().max().item()
    assert err <= TOL[dtype], err
