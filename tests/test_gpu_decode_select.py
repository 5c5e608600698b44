"""The selection's and the decode split's dispatch lines: sizes at the edges of each variant."""
import ctypes
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
    """Longest row of every workgroup size and chunk count, one more entry, and both sides of the 256 rows
    at which rows beyond 32768 entries change the workgroup size.  The selection is exact: no tolerance."""
    _check_selection(cuda, L, rows)


@pytest.mark.parametrize("L", [16384, 16385, 32768])
@pytest.mark.parametrize("rows", [512, 513])
def test_register_selection_on_both_sides_of_512_rows(cuda, L, rows):
    """Rows of 16385 to 32768 entries take workgroups of 1024 threads up to 512 rows and of 512 beyond."""
    _check_selection(cuda, L, rows)


def _check_selection(cuda, L, rows):
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L)
    base = (torch.rand(3, L, generator=gen) ** 4 * 512).round().half() / 512      # many ties
    k = max(1, L // 10)
    sc = base.to(cuda).repeat(math.ceil(rows / 3), 1)[:rows].contiguous()
    idx = kernels.topk_indices(sc, k).cpu()
    assert all(torch.equal(idx[r], idx[r % 3]) for r in range(rows))
    _check_rows(base, idx[:3], lambda r: k, lambda r: L, f"L={L}")


@pytest.mark.parametrize("H,G,L", [(32, 8, 1), (32, 8, 2047), (8, 8, 2049), (28, 4, 4096), (40, 8, 4097), (64, 4, 8192),
                                   (32, 8, 8193), (28, 4, 16384), (16, 2, 16385), (32, 8, 32768), (32, 8, 32769)])
@pytest.mark.parametrize("ragged", [False, True])
def test_anchor_selection_in_one_call(cuda, H, G, L, ragged):
    """kascade_decode_anchor_topk_call selects exactly the largest of the scores that the anchor pass
    pools by itself (checked against the oracle in test_gpu_decode): the two share the arithmetic, so
    there is no tolerance.  Row lengths at the edges of each pooling variant, groups of 1 to 16 heads."""
    from kascade_amd import _lib, kernels
    D, page, p = 128, 16, 10.0
    gen = torch.Generator().manual_seed(L + H)
    lens = [L, max(1, L // 3), max(1, L - 1)] if ragged else [L, L]
    B, pages = len(lens), math.ceil(L / page)
    q = torch.randn(B, H, D, generator=gen).half().to(cuda)
    kp = torch.randn(B * pages, page, G, D, generator=gen).half().to(cuda)
    bt = torch.randperm(B * pages, generator=gen).to(torch.int32).view(B, pages).to(cuda)
    seq = torch.tensor(lens, dtype=torch.int32, device=cuda)
    ns, stride = min(4, math.ceil(L / 64)), (L + 7) // 8 * 8
    glse = torch.empty(B, H, ns, device=cuda)
    sums, scores = torch.empty(B, H, device=cuda), torch.empty(B, H, stride, device=cuda)
    _, agg = kernels.decode_recompute(q, kp, kp, glse, None, sums, scores, 1, cache_seqlens=seq, block_table=bt,
                                      page_size=page, kv_len=L)
    want_sums = sums.clone()
    nsel = [math.ceil(int(p * n / 100) / 128) * 128 for n in lens] if ragged else [max(1, L // 10)] * B
    k = max(1, max(nsel))
    lib, ptr = _lib.init(), lambda t: None if t is None else t.data_ptr()
    idx = torch.full((B, G, k), -7, dtype=torch.int32, device=cuda)
    rows = torch.full_like(idx, -7)
    big = L > 32768
    per_row = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda).repeat_interleave(G) if big and ragged else None
    valid_d, nsel_d = per_row(lens), per_row(nsel)
    agg2 = torch.empty(B, G, stride, device=cuda, dtype=torch.float16) if big else None
    shape = ctypes.byref(_lib.Shape(G, D, kernels._ELEM[torch.float16], H // G))
    _lib.check(lib.kascade_decode_anchor_topk_call(
        shape, ptr(q), ptr(kp), None, ptr(seq), ptr(glse), None, ptr(sums), ptr(scores), None, ptr(agg2), ptr(idx), ptr(rows),
        B, L, stride, ns, 0, L, k, 5, p if ragged else 0.0, ptr(valid_d), ptr(nsel_d), None, ptr(bt), pages, page, None, None,
        None, None, torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(sums, want_sums)
    idx, pooled = idx.cpu(), agg.cpu()
    table = bt.cpu().long()
    for b in range(B):
        n, valid = nsel[b], lens[b]
        _check_rows(pooled[b], idx[b], lambda r: n, lambda r: valid, f"sequence {b}")
        assert bool((idx[b, :, n:] == 5).all())
        t = idx[b].long()
        inside = t < L
        want = table[b][(t.clamp(max=L - 1)) // page] * page + t % page
        assert torch.equal(rows[b].cpu().long()[inside], want[inside])


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


@pytest.mark.parametrize("heads,tokens", [(32, 3849), (32, 3850), (64, 5129), (64, 5130)])
def test_lists_on_both_sides_of_the_lone_split(cuda, heads, tokens):
    """Lists of 384 (512 from five query heads per KV head on) rows are gathered by one workgroup per
    KV head, longer ones by several: a reuse layer against the oracle on the anchor's own lists."""
    from types import SimpleNamespace
    from kascade_amd.strategy import EfficientKascadeStrategy
    G, D = 8, 128
    gen = torch.Generator().manual_seed(tokens)
    q = torch.randn(2, heads, 1, D, generator=gen).half()
    k, v = (torch.randn(2, G, tokens, D, generator=gen).half() for _ in range(2))
    s = EfficientKascadeStrategy([0], None, k=10, tile_size=32, head_mapping=[list(range(G)), [3] * G], register=False)
    for layer in (0, 1):
        o, _ = s.attention_forward(SimpleNamespace(layer_idx=layer), q.to(cuda), k.to(cuda), v.to(cuda), None, D ** -0.5)
    idx = s._topk_to_reuse.cpu()
    assert idx.shape[-1] == (384 if heads == 32 else 512) + (0 if tokens % 2 else 128)
    want = orc.reuse_decode(q[:, :, 0], k.transpose(1, 2), v.transpose(1, 2), idx, [3] * G, [idx.shape[-1]] * 2)
    assert_close(o[:, 0], want, "reuse output")


@pytest.mark.parametrize("H,G,L", [(32, 8, 2100), (8, 8, 700), (16, 1, 4200)])
@pytest.mark.parametrize("level", [0.0, -30.0, -45.0, -55.0])
def test_masked_scores_pool_to_nothing_in_one_call(cuda, H, G, L, level):
    """Tokens whose score is -inf for every head (a key with an infinite component): whole granules of 64,
    parts of some, a whole sequence -- while the other scores lie near ``level`` (log2 domain), so that a
    masked token's share must be 0 and not the least the score codes express.  Exactly the selection
    over the scores that the two-launch route pools; a masked token goes after every token above 0."""
    from kascade_amd import _lib, budgets, kernels
    D, B = 128, 2
    gen = torch.Generator().manual_seed(L)
    q = 1 + 0.1 * torch.randn(B, H, 1, D, generator=gen)
    k = level / (D ** 0.5 * orc.LOG2E) + 0.2 * torch.randn(B, G, L, D, generator=gen)
    masked = torch.zeros(B, L, dtype=torch.bool)
    masked[0, 64:192] = masked[0, 300:500] = masked[0, L - 70:] = True
    masked[1] = True
    k[..., 5][masked[:, None].expand(B, G, L)] = -float("inf")
    q, k = q.half().to(cuda), k.half().to(cuda)
    v = torch.randn(B, G, L, D, generator=gen).half().to(cuda)
    width = budgets.topk_width(L, 10)
    same = torch.arange(G, device=cuda, dtype=torch.int32)
    ns, stride = 3, (L + 7) // 8 * 8
    glse, part = torch.empty(B, H, ns, device=cuda), torch.empty(B, H, ns, D, device=cuda)
    sums, scores = torch.empty(B, H, device=cuda), torch.empty(B, H, stride, device=cuda)
    native = _lib.native()
    for layer in (0, 1):
        _, agg = kernels.decode_recompute(q[:, :, 0], k.transpose(1, 2), v.transpose(1, 2), glse, part, sums, scores, layer)
        assert bool((agg[:, :, :L][masked[:, None].expand(B, G, L).to(cuda)] == 0).all())
        want = kernels.topk_indices(agg[:, :, :L], width, fill_value=0)
        _, idx = native.hf_decode_anchor(native.Counters(), q, k, v, layer == 0, width, same)
        assert torch.equal(idx, want), f"layer {layer}"
        assert not bool(masked[0][idx[0].cpu().long()].any())


@pytest.mark.parametrize("H,G,L", [(64, 8, 18432), (64, 8, 18433), (28, 4, 20001), (32, 8, 24577), (4, 4, 32767), (32, 2, 32768)])
@pytest.mark.parametrize("ragged", [False, True])
def test_anchor_selection_with_and_without_buffers_for_two_launches(cuda, H, G, L, ragged):
    """Rows beyond kascade_pool_select_row are pooled and selected in two launches when the caller gives the
    buffers for it, in one otherwise: the same lists, cache rows and log-sums."""
    from kascade_amd import _lib, kernels
    D, page, p = 128, 16, 10.0
    lib = _lib.init()
    gen = torch.Generator(device=cuda).manual_seed(L)
    lens = [L, L // 3] if ragged else [L, L]
    B, pages = len(lens), math.ceil(L / page)
    assert (L > lib.kascade_pool_select_row(H // G, B * G)) == (L != 18432)
    q = torch.randn(B, H, D, generator=gen, device=cuda).half()
    kp = torch.randn(B * pages, page, G, D, generator=gen, device=cuda).half()
    bt = torch.arange(B * pages, dtype=torch.int32, device=cuda).view(B, pages)
    seq = torch.tensor(lens, dtype=torch.int32, device=cuda)
    ns, stride = 4, (L + 7) // 8 * 8
    nsel = [math.ceil(int(p * n / 100) / 128) * 128 for n in lens] if ragged else [L // 10] * B
    k = max(nsel)
    per_row = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda).repeat_interleave(G)
    agg = torch.empty(B, G, stride, device=cuda, dtype=torch.float16)
    shape, ptr = ctypes.byref(_lib.Shape(G, D, 0, H // G)), lambda t: None if t is None else t.data_ptr()
    got = []
    for buffers in ((None, None, None), (agg, per_row(lens) if ragged else None, per_row(nsel) if ragged else None)):
        glse, sums = torch.empty(B, H, ns, device=cuda), torch.empty(B, H, device=cuda)
        scores = torch.empty(B, H, stride, device=cuda)
        idx = torch.full((B, G, k), -7, dtype=torch.int32, device=cuda)
        rows = torch.full_like(idx, -7)
        _lib.check(lib.kascade_decode_anchor_topk_call(
            shape, ptr(q), ptr(kp), None, ptr(seq), ptr(glse), None, ptr(sums), ptr(scores), None, ptr(buffers[0]), ptr(idx),
            ptr(rows), B, L, stride, ns, 0, L, k, 5, p if ragged else 0.0, ptr(buffers[1]), ptr(buffers[2]), None, ptr(bt),
            pages, page, None, None, None, None, torch.cuda.current_stream().cuda_stream))
        torch.cuda.synchronize()
        got.append((idx, rows, sums))
    assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("H,G,L", [(8, 8, 700), (32, 8, 2100), (16, 1, 9001)])
def test_scores_beyond_the_codes_range_in_one_call(cuda, H, G, L):
    """bf16 scores around 1e19, where a sum of exponentials in 32 bits can come out as nothing, with tokens whose
    score overflows to -inf for some heads only: the lists are those of the two-launch route all the same."""
    from kascade_amd import _lib, kernels
    D, k_sel = 128, 128
    gen = torch.Generator().manual_seed(L)
    q, k = torch.randn(1, H, 1, D, generator=gen), torch.randn(1, G, L, D, generator=gen)
    q[:, ::2, :, 3], q[:, 1::2, :, 3] = 1e20, 1.0
    k[:, :, 100:300, 3] = -1e30
    q, k = q.bfloat16().to(cuda), k.bfloat16().to(cuda)
    glse, sums = torch.empty(1, H, 3, device=cuda), torch.empty(1, H, device=cuda)
    scores = torch.empty(1, H, (L + 7) // 8 * 8, device=cuda)
    _, agg = kernels.decode_recompute(q[:, :, 0], k.transpose(1, 2), k.transpose(1, 2), glse, None, sums, scores, 1)
    want = kernels.topk_indices(agg[:, :, :L], k_sel, fill_value=0)
    native = _lib.native()
    _, idx = native.hf_decode_anchor(native.Counters(), q, k, k, False, k_sel, torch.arange(G, device=cuda, dtype=torch.int32))
    assert torch.equal(idx, want)


@pytest.mark.parametrize("H,G,lens,ns", [(5, 1, [1], 1), (28, 4, [2047, 9], 3), (8, 8, [2048, 2049], 2), (16, 1, [2056, 1], 65),
                                         (40, 4, [6145, 2048, 4097], 70), (32, 8, [4096, 700], 64), (9, 1, [333], 5)])
@pytest.mark.parametrize("layer", [0, 1])
def test_pooling_launch_follows_the_scores_it_is_given(cuda, H, G, lens, ns, layer):
    """The pooled scores of an anchor pass from the 16-bit codes in its scratch and its log-sums: groups of 1 to 16 heads
    (not only multiples of the four that are requested together), lengths at the edges of a workgroup's 2048 tokens, more
    and fewer splits than a wavefront has lanes.  In float64; an fp32 sum of up to 16 exponentials whose arguments are
    below 32 in size is off by less than 2^-18, so one step of fp16 covers rounding and ties."""
    from kascade_amd import kernels
    D, page = 128, 16
    gen = torch.Generator().manual_seed(H + lens[0])
    B, L = len(lens), max(lens)
    pages, stride = math.ceil(L / page), (L + 7) // 8 * 8 + 2048
    q = torch.randn(B, H, D, generator=gen).half().to(cuda)
    kp = torch.randn(B * pages, page, G, D, generator=gen).half().to(cuda)
    bt = torch.randperm(B * pages, generator=gen).to(torch.int32).view(B, pages).to(cuda)
    seq = torch.tensor(lens, dtype=torch.int32, device=cuda)
    glse, part = torch.empty(B, H, ns, device=cuda), torch.empty(B, H, ns, D, device=cuda)
    sums, scores = torch.empty(B, H, device=cuda), torch.empty(B, H, stride, device=cuda)
    _, agg = kernels.decode_recompute(q, kp, kp, glse, part, sums, scores, layer, cache_seqlens=seq, block_table=bt,
                                      page_size=page, kv_len=L)
    torch.cuda.synchronize()
    agg = agg.cpu()
    codes = scores.cpu().view(torch.int16).view(B, H, 2 * stride)[..., :stride].to(torch.int32) & 0xFFFF
    refs = scores.cpu()[..., stride // 2:].double()
    total = torch.logsumexp(glse.cpu().double() * math.log(2.0), -1) / math.log(2.0)
    assert float((sums.cpu().double() - total).abs().max()) < 1e-5
    for b, n in enumerate(lens):
        ref = refs[b, :, :(n + 63) // 64].repeat_interleave(64, -1)[:, :n]
        p = torch.exp2(ref - codes[b, :, :n].double() / 2048.0 - total[b, :, None])
        want = p.view(G, H // G, n).sum(1)
        step = torch.clamp(want, min=2.0 ** -14) * 2.0 ** -10
        assert bool(((agg[b, :, :n].double() - want).abs() <= step).all())
        assert not bool(agg[b, :, n:].any())
