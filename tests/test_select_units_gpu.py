"""Block selection at sizes where the walks' work units change length (32, 64, 128 or 256 pairs of the forward and dQ walks, 64, 128 or
256 of the dK / dV walk), one token to either side of a line, against the CPU oracle."""

import pytest

from tests.test_select_gpu import test_select_fwd_bwd_matches_oracle as check

pytestmark = pytest.mark.gpu


# batch, heads, kv heads, tokens, d, block, slots; pairs = batch * kv heads * tokens * (slots + 1)
@pytest.mark.parametrize("b,hq,hk,n,d,B,S", [
    (1, 4, 2, 300, 128, 64, 5),                                   # 3600: units of 32 and 64 pairs
    (2, 8, 2, 3276, 64, 64, 4), (2, 8, 2, 3277, 64, 64, 4),       # 65520, 65540: dK / dV 64 -> 128
    (1, 16, 4, 6553, 64, 32, 4), (1, 16, 4, 6554, 64, 32, 4),     # 131060, 131080: forward 32 -> 64, dK / dV 128 -> 256
    (2, 8, 4, 3277, 128, 64, 4),                                  # 131080
    (2, 8, 4, 6553, 64, 64, 4), (2, 8, 4, 6554, 64, 64, 4),       # 262120, 262160: forward 64 -> 128
])
def test_units_of_every_length(b, hq, hk, n, d, B, S):
    check(b, hq, hk, n, d, B, S)
