"""Which decode projections run as one launch: the limits of the form that keeps x in registers (32 rows, K 2304)
and what stays one launch past them."""
import pytest

from lit_gpt._inference import proj_fused


@pytest.mark.parametrize("M,N,K,norm,gated,fused", [
    (1, 32000, 2304, True, False, True), (32, 7208, 2304, True, True, True), (32, 32000, 64, True, False, True),
    (33, 32000, 2304, True, False, False), (64, 7208, 2304, True, True, False), (33, 100, 2304, False, True, False),
    (33, 4096, 1024, True, False, True), (64, 4096, 1024, True, True, True), (64, 4097, 1024, True, False, False),
    (64, 4096, 1032, True, False, False),
    (1, 100, 2312, True, False, False), (4, 7680, 2560, True, True, False), (9, 7680, 2560, True, False, False),
    (32, 7680, 2560, True, True, False),
    (5, 7680, 2560, True, False, True), (8, 32000, 5120, True, False, True),  # the GEMV's slow rows
    (9, 9216, 3072, True, True, True), (16, 9216, 3072, True, True, True), (17, 9216, 3072, True, True, False),
    (9, 9240, 3080, True, True, False),
    (1, 2304, 7208, False, False, True), (64, 2304, 7208, False, False, True), (64, 2304, 2304, False, False, True),
])
def test_one_launch_where_x_is_not_streamed(M, N, K, norm, gated, fused):
    assert proj_fused(M, N, K, norm, gated) is fused
