"""Which prefill batches get room for partial states: the host's rule against measured times (us,
MI355X, whole calls with the append) of the uncut launch and of the split launch."""

import pytest

from kavor_amd.layers.attention import _may_split, _split_pays

# sequences, new tokens (all, longest), keys of the longest, query heads, kv heads; uncut, split
MEASURED = [
    ((3, 474, 300, 8492, 32, 8), 155.2, 62.7),    # turns of 17-300 tokens on 2048-8192 cached
    ((1, 2500, 2500, 10692, 16, 8), 254.9, 220.9),
    ((1, 1100, 1100, 1100, 16, 8), 37.1, 33.2),
    ((1, 2000, 2000, 2000, 16, 8), 59.0, 45.7),
    ((8, 1600, 200, 4296, 16, 8), 111.7, 85.7),   # eight on one shared prefix
    ((8, 2240, 500, 2548, 16, 8), 60.4, 52.4),    # ragged: 60-500 new on 0-2048
    ((4, 1800, 700, 3700, 16, 8), 81.0, 60.0),    # ragged: 200-700 new on 500-3000
    ((16, 256, 16, 8208, 64, 8), 207.9, 130.4),
    ((2, 1500, 750, 15750, 32, 8), 407.8, 411.4),
    ((3, 1500, 500, 15500, 32, 8), 406.7, 410.4),
    ((4, 1500, 375, 15375, 32, 8), 406.0, 408.7),
    ((2, 2000, 1000, 5096, 32, 8), 163.1, 165.2),
    ((4, 2800, 700, 2748, 16, 8), 84.7, 88.0),
    ((32, 3200, 100, 2148, 16, 8), 80.4, 83.1),   # short prompts on one shared prefix
    ((16, 1920, 120, 1144, 16, 8), 45.1, 46.9),
    ((8, 2000, 250, 1274, 16, 8), 47.5, 49.0),
    ((4, 2000, 500, 1012, 16, 8), 40.6, 43.2),
    ((2, 2048, 1024, 1024, 16, 8), 39.3, 40.7),
    ((4, 4096, 1024, 1024, 16, 8), 45.3, 48.5),
    ((3, 3900, 1300, 1300, 16, 8), 50.5, 54.3),
]


@pytest.mark.parametrize("batch,uncut,split", MEASURED)
def test_the_faster_launch_is_chosen(batch, uncut, split):
    num_seqs, _, max_q, max_k, hq, hkv = batch
    assert (_may_split(num_seqs, max_q, max_k, hq, hkv) and _split_pays(*batch)) == (split < uncut)
