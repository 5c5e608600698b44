"""The prompt kernels' dispatch lines: sizes on both sides of each, and tile remainders."""
import pytest
import torch

from oracle import kascade_oracle as orc
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L", [(1, 1), (16, 255), (16, 256), (16, 257), (17, 250), (13, 321)])
def test_log_sums_on_both_sides_of_the_unit_size(cuda, B, L):
    """32 queries per wavefront up to 512 units of 64 queries, 64 beyond (8 KV heads).  Tolerance as
    for the log-sums elsewhere: fp32 sums of exponentials of fp32-accumulated fp16 products."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L)
    q = torch.randn(1, L, 32, 128, generator=gen).half()
    k = torch.randn(1, L, 8, 128, generator=gen).half()
    _, want = orc.dense_prefill(q, k, k)
    got = kernels.prefill_recompute1(q.to(cuda).repeat(B, 1, 1, 1), k.to(cuda).repeat(B, 1, 1, 1))
    assert_close(got, want.repeat(B, 1, 1), f"log_sum {B}x{L}", atol=2e-3, rtol=1e-4)
