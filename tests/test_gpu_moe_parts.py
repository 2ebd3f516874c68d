"""Few-token routed steps, whose grouped GEMVs cut a row tile's blocks into
parts (whole-step entry point), against the oracle.
"""
import pytest

from test_gpu_moe import TIGHT, batch_case
from conftest import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,H,I,shared", [
    (1, 8, 2, 1792, 768, True),    # 7 and 3 blocks: parts of unequal length, rows too short for four
    (1, 4, 1, 256, 256, False),    # one block: one part
    (1, 64, 8, 2560, 2048, True),  # 10 and 8 blocks in four and up to four parts
    (2, 16, 4, 2048, 512, True),   # 8 and 2 blocks
    (9, 64, 8, 1024, 1024, True),  # more items than wavefronts for some tensors, two shared segments
    (70, 64, 8, 512, 512, True),   # a third round and more slots than the parts' room
])
def test_parts_match_oracle(gpu, T, E, K, H, I, shared):
    Y, ref = batch_case(gpu, 97, T, E, K, H, I, 0, shared)[:2]
    for t in range(T):
        assert rel_err(Y[t], ref[t]) < TIGHT, t
