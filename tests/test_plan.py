"""Plans of the E-steps, queried without a GPU."""

import pytest

from routes import plan_info


# The widest plans that screen (the rows' block bounds fill LDS), and ordinary ones.
@pytest.mark.parametrize("model,K,D,state,word", [("iso", 4352, 32, 16, 4), ("iso", 4300, 2, 16, 4),
                                                  ("iso", 1024, 128, 16, 4), ("diag", 3840, 32, 8, 8),
                                                  ("diag", 1792, 96, 8, 8)])
@pytest.mark.parametrize("N", [1_000_000, 2_030_000_000, (1 << 31) - 300])
def test_slab_offsets_fit_32_bits(model, K, D, state, word, N):
    """The gathering pass 2 reads a slab's row state and need words at 32-bit byte offsets."""
    screen, _, _, _, rows, nslab = plan_info(model, N, K, D)
    assert screen
    KB = -(-K // 32)
    assert rows % 32 == 0 and (nslab - 1) * rows < N <= nslab * rows
    assert rows * state < 2 ** 31
    assert (rows // 32) * KB * word < 2 ** 31
