"""What hgemm_auto plans at sizes where two routes meet (no launch, no GPU)."""
import pytest


@pytest.mark.parametrize("M", [129, 150, 192])
@pytest.mark.parametrize("N", [18432, 28672, 57344])
def test_no_copies_below_the_one_row_rule(hgemm_lib, M, N):
    """K just short of 2048: the copies' padded K would be the first the 192x128 one-row rule covers."""
    for K in range(1992, 2048, 8):
        assert hgemm_lib.auto_workspace_bytes(M, N, K)["operands"] == 0, K
