"""The selection's and the decode split's dispatch lines: sizes at the edges of each variant."""
import math

import pytest
import torch

from oracle import kascade_oracle as orc
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu


def _check_rows(scores, idx, n_of, valid_of, what):
    for r in range(scores.shape[0]):
        n, valid = n_of(r), valid_of(r)
        if valid <= n:      # every token, then the positions behind them
            assert torch.equal(idx[r, :n], torch.arange(n, dtype=torch.int32)), f"{what} row {r}"
            continue
        ok, _, msg = orc.topk_agreement(scores[r], idx[r], n, valid, ulps=0.0)
        assert ok, f"{what} row {r}: {msg}"
        assert bool((idx[r, 1:n] > idx[r, :n - 1]).all()), f"{what} row {r}: not ascending"


@pytest.mark.parametrize("L", [1, 8, 511, 513, 2048, 2049, 4096, 4097, 8193, 16384, 16385, 32768, 32769, 65536])
@pytest.mark.parametrize("rows", [3, 257])
def test_register_selection_edges(cuda, L, rows):
    """Longest row of every workgroup size and chunk count, one more entry, and both sides of the
    row count at which long rows change the workgroup size.  The selection is exact: no tolerance."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L)
    base = (torch.rand(3, L, generator=gen) ** 4 * 512).round().half() / 512      # many ties
    k = max(1, L // 10)
    sc = base.to(cuda).repeat(math.ceil(rows / 3), 1)[:rows].contiguous()
    idx = kernels.topk_indices(sc, k).cpu()
    assert all(torch.equal(idx[r], idx[r % 3]) for r in range(rows))
    _check_rows(base, idx[:3], lambda r: k, lambda r: L, f"L={L}")


@pytest.mark.parametrize("seqlens,ns", [([1024], 1), ([1025], 1), ([2048, 1], 1), ([2049, 64], 1), ([255, 257, 4096], 2),
                                        ([63, 64, 65, 128, 129], 1), ([1500, 40] * 10, 4), ([700] * 20, 4)])
def test_split_strips_and_direct_output(cuda, seqlens, ns):
    """Rows per split on both sides of each strip width, splits whose wavefronts own nothing, one split
    that writes the result itself, and batches on both sides of the in-kernel numbering's line (20
    sequences of four splits).  Tolerance: assert_close's (fp16 results, fp32 accumulation)."""
    from kascade_amd import kernels, workloads
    H, G, D = 32, 8, 128
    w = workloads.paged_decode_inputs(seqlens, seed=ns + len(seqlens), device="cpu", peaked=True)
    kc = orc.paged_to_contiguous(w.k_pages, w.block_table, seqlens)
    vc = orc.paged_to_contiguous(w.v_pages, w.block_table, seqlens)
    want, lse = orc.dense_decode(w.q, kc, vc, seqlens)
    B, L = len(seqlens), max(seqlens)
    q, kp, vp, lens, bt = (t.to(cuda) for t in (w.q, w.k_pages, w.v_pages, w.seqlens, w.block_table))
    for sync in (None, torch.zeros(B * G, dtype=torch.int32, device=cuda)):
        glse, part = torch.empty(B, H, ns, device=cuda), torch.empty(B, H, ns, D, device=cuda)
        got = kernels.decode_dense_paged(q, kp, vp, lens, glse, part, bt, w.page_size, sync=sync)
        assert_close(got, want, f"dense, merged in launch={sync is not None}")
        sums, stride = torch.empty(B, H, device=cuda), (L + 7) // 8 * 8
        scores = torch.empty(B, H, stride, device=cuda)
        for layer in (0, 1):
            o, agg = kernels.decode_recompute(q, kp, vp, glse, part, sums, scores, layer, cache_seqlens=lens, block_table=bt,
                                              page_size=w.page_size, sync=sync)
            assert_close(sums, lse * orc.LOG2E, "row_sums", atol=2e-3, rtol=1e-4)
            assert_close(agg.cpu()[:, :, :L], orc.pooled_decode_scores(w.q, kc, seqlens), "pooled scores", atol=2e-6, rtol=2e-3)
            if layer == 0:
                assert_close(o, want, "anchor-0 output")
        if sync is not None:
            assert int(sync.abs().sum()) == 0
