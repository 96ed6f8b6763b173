"""The attention prologue around the rule from which a wave takes three or four heads
of a token: a last run that is not full, runs that hold query and key, or key and
value heads, a head size that is not a multiple of 64, the last token count with one
head per wave, and rotations of up to 64 elements, of two more and of a whole head.  The check is test_gpu_prologue.py's: equal to the unfused
chain bit for bit, and close to the oracle."""
import pytest

from test_gpu_prologue import test_prologue_matches_unfused_chain_and_oracle as check

TEXT = (11, 11, 10, 0)
CASES = [
    # tokens, start, cap, layers, layer, heads, kv_heads, d, n_dims, sections, explicit positions
    (255, 1, 256, 1, 0, 8, 2, 256, 64, TEXT, False),
    (256, 10, 270, 2, 1, 8, 2, 256, 64, TEXT, False),
    (341, 3, 344, 1, 0, 8, 2, 256, 64, TEXT, False),        # 4092 heads, one per wave
    (342, 10, 360, 2, 1, 8, 2, 256, 64, TEXT, False),       # 4104 heads, three per wave
    (300, 0, 300, 1, 0, 7, 1, 96, 64, TEXT, True),
    (456, 0, 456, 1, 0, 7, 1, 96, 64, TEXT, True),          # 9 heads a token, three per wave
    (256, 2, 258, 1, 0, 8, 2, 256, 256, (44, 44, 40, 0), False),  # the whole head rotates
    (17, 2, 19, 1, 0, 8, 2, 256, 66, (11, 11, 11, 0), True),      # one pair past 64 elements
    (261, 5, 266, 1, 0, 10, 5, 256, 192, (24, 20, 12, 8), True),  # 20 heads, four per wave
    (256, 3, 259, 1, 0, 9, 3, 128, 128, (24, 20, 12, 8), True),   # 15 heads, a run of three left
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_prologue_runs_of_heads(hip_ctx, case):
    check(hip_ctx, case)
