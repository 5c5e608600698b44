"""The prompt kernels' dispatch lines: sizes on both sides of each, and tile remainders."""
import math

import pytest
import torch

from oracle import kascade_oracle as orc
from tests.helpers import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L", [(1, 1), (16, 255), (16, 256), (16, 257), (17, 250), (13, 321)])
def test_log_sums_on_both_sides_of_the_unit_size(cuda, B, L):
    """Batches of short prompts around 512 units of 64 queries (8 KV heads).  Tolerance as
    for the log-sums elsewhere: fp32 sums of exponentials of fp32-accumulated fp16 products."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L)
    q = torch.randn(1, L, 32, 128, generator=gen).half()
    k = torch.randn(1, L, 8, 128, generator=gen).half()
    _, want = orc.dense_prefill(q, k, k)
    got = kernels.prefill_recompute1(q.to(cuda).repeat(B, 1, 1, 1), k.to(cuda).repeat(B, 1, 1, 1))
    assert_close(got, want.repeat(B, 1, 1), f"log_sum {B}x{L}", atol=2e-3, rtol=1e-4)


@pytest.mark.parametrize("L", [33, 129, 517, 897, 1300, 2048, 2049])
@pytest.mark.parametrize("heads,G,D", [(32, 8, 128), (28, 4, 64)])
def test_pooled_scores_do_not_depend_on_the_key_parts(cuda, L, heads, G, D):
    """Small calls cut a tile's keys into parts, a batch of copies of the same prompt does not: the same
    bits, the invalid positions' fill included, and the oracle's scores to fp16 rounding."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L + D)
    q = torch.randn(1, L, heads, D, generator=gen).half()
    k = torch.randn(1, L, G, D, generator=gen).half()
    T, B = (L + 31) // 32, 512 // (G * ((L + 31) // 32)) + 1
    log_sum = kernels.prefill_recompute1(q.to(cuda), k.to(cuda))

    def pooled(n):
        qd, kd = q.to(cuda).repeat(n, 1, 1, 1), k.to(cuda).repeat(n, 1, 1, 1)
        out = torch.full((n, G, T, L), 7.0, device=cuda, dtype=torch.float16)
        kernels.prefill_aggregate(qd, kd, log_sum.repeat(n, 1, 1), out, fill_invalid=True)
        return out
    one, many = pooled(1), pooled(B)
    assert all(torch.equal(one[0], m) for m in many)
    if L <= 1300:
        want = orc.pooled_prefill_scores(q, k, 32).reshape(G, T, L).float()
        keys = torch.arange(L).view(1, 1, L) < 32 * torch.arange(T).view(1, T, 1)
        got = one[0].float().cpu()
        assert bool((got[~keys.expand_as(got)] == -float("inf")).all())
        # an fp16 rounding of the sum plus the fp32 noise of 128 exponentials
        assert_close(got[keys.expand_as(got)], want[keys.expand_as(want)], "pooled scores", atol=1e-4, rtol=2e-3)


@pytest.mark.parametrize("B,n,start", [(16, 256, 256), (16, 250, 256), (16, 256, 0), (17, 225, 96)])
def test_chunk_log_sums_do_not_depend_on_the_unit_size(cuda, B, n, start):
    """A chunk's log-sums over the paged cache, in a batch of about 512 units (64 queries per wavefront
    where the units are equally long) and alone (32): the same bits, and the oracle's values."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(n)
    L, page = start + n, 16
    q = torch.randn(1, L, 32, 128, generator=gen).half()
    k = torch.randn(1, L, 8, 128, generator=gen).half()
    per = (L + page - 1) // page
    pages = torch.zeros(per * page, 8, 128, dtype=torch.float16)
    pages[:L] = k[0]
    order = torch.randperm(per, generator=gen)
    kp = torch.empty(per, page, 8, 128, dtype=torch.float16)
    kp[order] = pages.view(per, page, 8, 128)
    kp = kp.to(cuda)

    def log_sum(b):
        table = order.to(torch.int32).repeat(b, 1).to(cuda)
        return kernels.prefill_chunk_dense(q[:, start:].repeat(b, 1, 1, 1).to(cuda), kp, kp, table, start,
                                           page_size=page, with_output=False)[0]
    one, many = log_sum(1), log_sum(B)
    assert all(torch.equal(one[0], m) for m in many)
    _, want = orc.dense_prefill(q, k, k)
    assert_close(one, want[:, start:], "chunk log_sum", atol=2e-3, rtol=1e-4)


def _paged_copies(k, page, gen, B, cuda):
    """k [1,L,G,D] in shuffled pages that B sequences share: (pages, block table)."""
    L, G, D = k.shape[1:]
    per = (L + page - 1) // page
    rows = torch.zeros(per * page, G, D, dtype=k.dtype)
    rows[:L] = k[0]
    order = torch.randperm(per, generator=gen)
    pages = torch.empty(per, page, G, D, dtype=k.dtype)
    pages[order] = rows.view(per, page, G, D)
    return pages.to(cuda), order.to(torch.int32).repeat(B, 1).to(cuda)


# units of 64 queries: 440 and 448, 512 and 520 (about equal lengths), 640 twice (equal, spread), 648, 768 and 800
# (short), 792 (whole prompts)
@pytest.mark.parametrize("B,n,start", [(11, 320, 320), (14, 256, 256), (16, 256, 256), (13, 320, 320), (10, 512, 1536),
                                       (5, 1024, 1024), (27, 192, 1888), (24, 256, 256), (25, 256, 256), (3, 2049, 0)])
def test_log_sums_have_the_same_bits_on_every_line_of_the_unit_size(cuda, B, n, start):
    """A batch of copies, whatever unit size the rule takes for it, against one of them alone (32 queries
    per wavefront): the same bits, over the paged cache and, from position 0, for whole prompts."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(n + start)
    q = torch.randn(1, start + n, 32, 128, generator=gen).half()
    k = torch.randn(1, start + n, 8, 128, generator=gen).half()
    kp, table = _paged_copies(k, 16, gen, B, cuda)
    qd = q[:, start:].to(cuda)
    one = kernels.prefill_chunk_dense(qd, kp, kp, table[:1], start, page_size=16, with_output=False)[0]
    many = kernels.prefill_chunk_dense(qd.repeat(B, 1, 1, 1), kp, kp, table, start, page_size=16, with_output=False)[0]
    assert all(torch.equal(one[0], m) for m in many)
    if start == 0:
        assert torch.equal(one, kernels.prefill_recompute1(qd, k.to(cuda)))
        many = kernels.prefill_recompute1(qd.repeat(B, 1, 1, 1), k.to(cuda).repeat(B, 1, 1, 1))
        assert all(torch.equal(one[0], m) for m in many)
    _, want = orc.dense_prefill(q, k, k)
    assert_close(one, want[:, start:], "log_sum", atol=2e-3, rtol=1e-4)


def test_wide_log_sum_units_of_sequences_at_different_positions(cuda):
    """512 units of 64 queries over a paged cache, each sequence with a start and a row count of its own
    (none, a part of a unit, remainders): every sequence's rows have the bits of a call of its own, and
    rows that belong to no sequence are not written."""
    from kascade_amd import _lib, kernels
    B, n, top = 16, 256, 256
    gen = torch.Generator().manual_seed(7)
    starts = [top, 0, 32, 224, 96, 256, 160, 64] * 2
    lens = [256, 256, 1, 33, 64, 0, 127, 255, 65, 31, 250, 128, 0, 192, 200, 96]
    k = torch.randn(1, top + n, 8, 128, generator=gen).half()
    kp, table = _paged_copies(k, 16, gen, B, cuda)
    q = torch.randn(B, n, 32, 128, generator=gen).half().to(cuda)
    at = lambda v: torch.tensor(v, dtype=torch.int32, device=cuda)
    got, qs, ql = torch.full((B, n, 32), 7.0, device=cuda), at(starts), at(lens)
    _lib.check(_lib.init().kascade_prefill_chunk_dense_call(
        q.data_ptr(), kp.data_ptr(), None, got.data_ptr(), None, B, top, n, _lib.Strides(*q.stride()[:3]), table.data_ptr(),
        table.shape[1], 16, kp.shape[0], 0, qs.data_ptr(), ql.data_ptr(), torch.cuda.current_stream().cuda_stream))
    for b in range(B):
        assert bool((got[b, lens[b]:] == 7.0).all())
        if lens[b]:
            own = kernels.prefill_chunk_dense(q[b:b + 1, :lens[b]], kp, kp, table[b:b + 1], starts[b], page_size=16,
                                              with_output=False)[0]
            assert torch.equal(got[b, :lens[b]], own[0]), f"sequence {b}"


@pytest.mark.parametrize("page", [4, 8, 64])
@pytest.mark.parametrize("heads,G,D,dtype", [(32, 8, 128, torch.float16), (14, 2, 64, torch.bfloat16)])
def test_pooled_scores_over_pages_of_every_size(cuda, page, heads, G, D, dtype):
    """Tiles of a chunk read their keys through 64 block-table entries at a time (256 tokens with the smallest
    pages; at head_dim 64 a load then covers two pages): the bits of the whole prompt over a strided cache,
    for chunks whose keys start and end in different groups of entries."""
    from kascade_amd import kernels
    L = 1300
    gen = torch.Generator().manual_seed(page + D)
    q = torch.randn(1, L, heads, D, generator=gen).to(dtype).to(cuda)
    k = torch.randn(1, L, G, D, generator=gen).to(dtype)
    kp, table = _paged_copies(k, page, gen, 1, cuda)
    k = k.to(cuda)
    log_sum = kernels.prefill_recompute1(q, k)
    whole = torch.empty(1, G, (L + 31) // 32, L, device=cuda, dtype=torch.float16)
    kernels.prefill_aggregate(q, k, log_sum, whole, fill_invalid=True)
    for start, end in ((0, 96), (96, 512), (512, 1300), (1280, 1300)):
        got = torch.empty(1, G, (end - start + 31) // 32, end, device=cuda, dtype=torch.float16)
        kernels.prefill_chunk_aggregate(q[:, start:end], kp, log_sum[:, start:end].contiguous(), got, table, start, page,
                                        fill_invalid=True)
        assert torch.equal(got, whole[:, :, start // 32:(end + 31) // 32, :end]), f"rows {start}..{end}"


@pytest.mark.parametrize("page", [4, 8, 128, 256])
@pytest.mark.parametrize("heads,G,D,dtype", [(32, 8, 128, torch.float16), (14, 2, 64, torch.bfloat16), (32, 8, 64, torch.float16)])
def test_attention_over_pages_of_every_size(cuda, page, heads, G, D, dtype):
    """Pages smaller than a tile (64 keys, 128 at head_dim 64), as large and larger: chunks that start in the middle of
    a page and end inside a tile have the bits of the whole prompt over a strided cache, dense, log-sums alone and
    sparse (with and without log-sums)."""
    from kascade_amd import budgets, kernels
    L, p = 1300, 10
    gen = torch.Generator().manual_seed(page + D)
    q = torch.randn(1, L, heads, D, generator=gen).to(dtype).to(cuda)
    k, v = (torch.randn(1, L, G, D, generator=gen).to(dtype) for _ in range(2))
    kp, table = _paged_copies(k, page, gen, 1, cuda)
    vp = torch.empty_like(kp)
    rows = torch.zeros(kp.shape[0] * page, G, D, dtype=dtype)
    rows[:L] = v[0]
    vp[table[0].long()] = rows.view(-1, page, G, D).to(cuda)
    k, v = k.to(cuda), v.to(cuda)
    log_sum, out = kernels.prefill_recompute0(q, k, v)
    T, W = (L + 31) // 32, budgets.topk_width(L, p)
    idx = torch.zeros(1, G, T, W, dtype=torch.int32)
    for t in range(1, T):
        n = min(32 * t, W)
        for g in range(G):
            idx[0, g, t, :n] = torch.randperm(32 * t, generator=gen)[:n].sort().values
    idx = idx.to(cuda)
    maps = torch.arange(G - 1, -1, -1, dtype=torch.int32, device=cuda)
    sparse, sparse_sums = kernels.prefill_reuse(q, k, v, idx, maps, float(p), True, return_log_sum=True)
    sparse_alone = kernels.prefill_reuse(q, k, v, idx, maps, float(p), True)
    for start, end in ((0, 96), (96, 500), (480, 1300), (1280, 1300)):
        qc = q[:, start:end]
        sums, o = kernels.prefill_chunk_dense(qc, kp, vp, table, start, page)
        assert torch.equal(sums, log_sum[:, start:end]) and torch.equal(o, out[:, start:end]), f"rows {start}..{end}"
        alone, _ = kernels.prefill_chunk_dense(qc, kp, vp, table, start, page, with_output=False)
        assert torch.equal(alone, sums), f"log-sums alone, rows {start}..{end}"
        width = budgets.topk_width(end, p)
        lists = kernels.translate_indices(idx[:, :, start // 32:(end + 31) // 32, :width].contiguous(), table, end, page)
        o, sums = kernels.prefill_chunk_reuse(qc, kp, vp, lists, maps, float(p), end > 128, table, start, page,
                                              return_log_sum=True)
        assert torch.equal(o, sparse[:, start:end]) and torch.equal(sums, sparse_sums[:, start:end]), f"sparse rows {start}..{end}"
        o = kernels.prefill_chunk_reuse(qc, kp, vp, lists, maps, float(p), end > 128, table, start, page)
        assert torch.equal(o, sparse_alone[:, start:end]), f"sparse rows {start}..{end}, no log-sums"


@pytest.mark.parametrize("L", [1, 15, 16, 17, 33, 47, 64, 65, 95, 129, 260])
@pytest.mark.parametrize("heads,G,dtype", [(32, 8, torch.float16), (7, 1, torch.bfloat16)])
def test_dense_rows_at_the_edges_of_query_and_key_blocks(cuda, L, heads, G, dtype):
    """Products of 16 queries whose exponentials are added up as those of 32: the log-sums have the bits of the pass
    for log-sums alone, outputs and log-sums are the oracle's (outputs to a rounding of the probabilities and one of the
    result)."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(L)
    q = torch.randn(2, L, heads, 128, generator=gen).to(dtype)
    k, v = (torch.randn(2, L, G, 128, generator=gen).to(dtype) for _ in range(2))
    k[:, 0] *= 3   # a reference that later tiles lie below, and above
    k[:, L // 2] *= 5
    want, want_sums = orc.dense_prefill(q, k, v)
    log_sum, out = kernels.prefill_recompute0(q.to(cuda), k.to(cuda), v.to(cuda))
    assert torch.equal(log_sum, kernels.prefill_recompute1(q.to(cuda), k.to(cuda)))
    assert_close(log_sum, want_sums, f"log-sums L={L}", atol=2e-3, rtol=1e-4)
    step = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7   # |v| reaches 4.5: two half steps of it
    assert_close(out, want, f"outputs L={L}", atol=4.5 * step, rtol=step)


@pytest.mark.parametrize("heads,G,D,dtype", [(32, 8, 128, torch.float16), (32, 8, 128, torch.bfloat16), (14, 2, 64, torch.float16)])
@pytest.mark.parametrize("batch", [1, 9])
def test_log_sums_alone_follow_late_maxima(cuda, batch, heads, G, D, dtype):
    """The pass for log-sums alone forms a tile's maximum only where the tile's sums ask for it: scores that
    rise step by step far behind the first tiles, by less and by more than the reference may lag and once beyond the
    range of the exponentials, give the bits of the pass with an output and the log-sum of float64.  Nine sequences
    of 32 heads take units of 64 queries."""
    from kascade_amd import kernels
    L = 4200 if batch == 1 else 1500
    gen = torch.Generator().manual_seed(D + batch)
    q = torch.randn(batch, L, heads, D, generator=gen).to(dtype).to(cuda)
    k = torch.randn(batch, L, G, D, generator=gen)
    for at, size in ((1, 3.0), (700, 6.0), (1100, 12.0), (1101, 24.0), (1290, 200.0)):
        k[:, at] *= size
    k = k.to(dtype).to(cuda)
    alone = kernels.prefill_recompute1(q, k)
    log_sum, _ = kernels.prefill_recompute0(q, k, k)
    assert torch.equal(alone, log_sum)
    b = batch - 1
    rows = torch.tensor([0, 1, 63, 64, 699, 700, 1023, 1099, 1101, 1289, 1290, 1299, L - 1], device=cuda)
    for h in (0, heads - 1):
        s = (q[b, rows, h].double() @ k[b, :, h // (heads // G)].double().t().contiguous()) * D ** -0.5
        s.masked_fill_(torch.arange(L, device=cuda)[None, :] > rows[:, None], float("-inf"))
        want = torch.logsumexp(s, 1) / 0.6931471805599453
        # scores are fp32 sums of D products of up to 200 x 4 x 4, the log-sum has 24 bits: 1e-6 of the largest
        bound = 1e-6 * s.masked_fill(s.isinf(), 0).abs().amax(1) / 0.69 + 4e-6 * want.abs() + 1e-5
        assert ((alone[b, rows, h].double() - want).abs() <= bound).all()


@pytest.mark.parametrize("gs", [1, 2, 3, 5, 6, 7])
@pytest.mark.parametrize("G,D,L", [(8, 128, 700), (4, 64, 1063), (3, 128, 31)])
def test_spare_head_slots_change_no_head(cuda, gs, G, D, L):
    """Groups that fill no whole four head slots leave wavefronts without a head.  Against the same call whose groups
    are filled up with copies of their last head (log-sum +inf in pooling: exp2(-inf) = 0 each): the same bits."""
    from kascade_amd import budgets, kernels
    gen = torch.Generator().manual_seed(10 * gs + L)
    q = torch.randn(2, L, G, gs, D, generator=gen).half()
    full = (gs + 3) // 4 * 4
    qf = torch.cat([q] + [q[:, :, :, -1:]] * (full - gs), dim=3).flatten(2, 3).to(cuda)
    q = q.flatten(2, 3).to(cuda)
    k, v = (torch.randn(2, L, G, D, generator=gen).half().to(cuda) for _ in range(2))

    def real(x):   # [B,L,G*full,...] without the copies
        return x.unflatten(2, (G, full))[:, :, :, :gs].flatten(2, 3)
    ls, out = kernels.prefill_recompute0(q, k, v)
    lsf, outf = kernels.prefill_recompute0(qf, k, v)
    assert torch.equal(ls, real(lsf)) and torch.equal(out, real(outf))
    assert torch.equal(kernels.prefill_recompute1(q, k), real(kernels.prefill_recompute1(qf, k)))

    T = (L + 31) // 32
    sc, scf = (torch.zeros(2, G, T, L, device=cuda, dtype=torch.float16) for _ in range(2))
    lsf = lsf.unflatten(2, (G, full)).clone()
    lsf[:, :, :, gs:] = float("inf")
    kernels.prefill_aggregate(q, k, ls, sc)
    kernels.prefill_aggregate(qf, k, lsf.flatten(2, 3).contiguous(), scf)
    assert torch.equal(sc, scf)

    width = budgets.topk_width(L, 10)
    valid, nsel = budgets.prefill_tile_budgets(L, 32, 10, True, width)
    idx = kernels.topk_indices(sc, width, valid_len=torch.tensor(valid, dtype=torch.int32, device=cuda),
                               n_sel=torch.tensor(nsel, dtype=torch.int32, device=cuda))
    hm = torch.arange(G, dtype=torch.int32, device=cuda).flip(0)
    assert torch.equal(kernels.prefill_reuse(q, k, v, idx, hm, 10.0, True),
                       real(kernels.prefill_reuse(qf, k, v, idx, hm, 10.0, True)))


@pytest.mark.parametrize("gs", [5, 8, 11, 16])
@pytest.mark.parametrize("G,D,L", [(8, 128, 161), (4, 64, 417), (3, 128, 1030), (1, 64, 129)])
def test_pooled_scores_add_up_over_the_sub_groups(cuda, gs, G, D, L):
    """Query heads are pooled four at a time and later launches add to the scores of the earlier ones.  Against launches
    over each sub-group alone: rounded to fp16 once per sub-group in either form, so half a step of a part, of the sum up
    to it and of the whole for every sub-group after the first (a step: 2^-10 of the value, 2^-24 at least)."""
    from kascade_amd import kernels
    gen = torch.Generator().manual_seed(gs + L)
    q = torch.randn(2, L, G, gs, D, generator=gen).half().to(cuda)
    k, v = (torch.randn(2, L, G, D, generator=gen).half().to(cuda) for _ in range(2))
    ls, _ = kernels.prefill_recompute0(q.flatten(2, 3).contiguous(), k, v)
    parts = ls.unflatten(2, (G, gs))
    T = (L + 31) // 32

    def pooled(h0, h1):
        sc = torch.full((2, G, T, L), 7.0, device=cuda, dtype=torch.float16)   # what a buffer holds before does not count
        kernels.prefill_aggregate(q[:, :, :, h0:h1].flatten(2, 3).contiguous(), k,
                                  parts[:, :, :, h0:h1].flatten(2, 3).contiguous(), sc, fill_invalid=True)
        return sc.double()
    got = pooled(0, gs)
    want, slack = torch.zeros_like(got), torch.zeros_like(got)
    for h0 in range(0, gs, 4):
        part = pooled(h0, min(h0 + 4, gs))
        want = want + part
        slack = slack + (part.abs() + want.abs() + got.abs()) * 2.0 ** -11 + 2.0 ** -24
    inside = torch.isfinite(got)
    assert torch.equal(inside, torch.isfinite(want)) and bool(inside.any())
    assert bool(((got - want).abs()[inside] <= slack[inside]).all())


# 256 units are cut in halves, 264 (or more) are not: copies of a prompt, and the same prompt over the paged cache
@pytest.mark.parametrize("heads,G,D,L,copies,dtype", [
    (32, 8, 128, 1024, 2, torch.float16), (32, 8, 128, 517, 2, torch.bfloat16), (28, 4, 128, 300, 7, torch.float16),
    (14, 2, 64, 2000, 2, torch.bfloat16), (8, 8, 128, 700, 2, torch.float16), (24, 8, 64, 129, 7, torch.float16),
    (5, 1, 128, 200, 19, torch.float16), (32, 2, 128, 161, 6, torch.bfloat16)])
def test_sparse_rows_do_not_depend_on_the_cut_of_a_unit(cuda, heads, G, D, L, copies, dtype):
    """Sparse units in halves (16 queries per wavefront, two head slots per workgroup) and whole ones: the same bits,
    with empty slots in one half or in both and blocks that end inside either 16 queries."""
    from kascade_amd import budgets, kernels
    p = 10
    gen = torch.Generator().manual_seed(L + heads)
    q = torch.randn(1, L, heads, D, generator=gen).to(dtype).to(cuda) * 2   # references that move behind the first tile
    k, v = (torch.randn(1, L, G, D, generator=gen).to(dtype) for _ in range(2))
    kp, table = _paged_copies(k, 16, gen, 1, cuda)
    rows = torch.zeros(kp.shape[0] * 16, G, D, dtype=dtype)
    rows[:L] = v[0]
    vp = torch.empty_like(kp)
    vp[table[0].long()] = rows.view(-1, 16, G, D).to(cuda)
    T, W = (L + 31) // 32, budgets.topk_width(L, p)
    idx = torch.zeros(1, G, T, W, dtype=torch.int32)
    for t in range(1, T):
        n = min(32 * t, W)
        for g in range(G):
            idx[0, g, t, :n] = torch.randperm(32 * t, generator=gen)[:n].sort().values
    maps = torch.arange(G - 1, -1, -1, dtype=torch.int32, device=cuda)
    units = T * G * -(-heads // G // 4)
    assert units <= 256 < units * copies
    kd, vd, idx = k.to(cuda), v.to(cuda), idx.to(cuda)
    one = kernels.prefill_reuse(q, kd, vd, idx, maps, float(p), True)
    many = kernels.prefill_reuse(*(x.repeat(copies, 1, 1, 1) for x in (q, kd, vd, idx)), maps, float(p), True)
    assert all(torch.equal(one[0], m) for m in many)
    lists = kernels.translate_indices(idx.contiguous(), table, L, 16)
    assert torch.equal(kernels.prefill_chunk_reuse(q, kp, vp, lists, maps, float(p), True, table, 0, 16), one)
    want = orc.reuse_prefill(q.cpu(), k, v, idx.cpu(), maps.tolist(), 32, True, float(p))
    atol, rtol = (2e-3, 1e-2) if dtype == torch.float16 else (1.6e-2, 2e-2)   # one rounding of P and of the output
    assert_close(one, want, "sparse rows", atol=atol, rtol=rtol)


def _anchor_inputs(cuda, gen, heads, G, D, L, B, dtype):
    q = torch.randn(B, L, heads, D, generator=gen).to(dtype).to(cuda)
    k = torch.randn(B, L, G, D, generator=gen).to(dtype)
    k[:, 0] += 1.0
    k[:, 5:40] = k[:, 4:5]   # equal keys: ties
    return q, k


# Units and key tiles on both sides of each line of the rule (kascade_prefill_pool_selects, the last column), with tails of every
# kind: up to 192 units with 6 tiles and with 7, 216 and 256 units, head_dim 64 with 8 and 9 tiles; up to 448 units with 16 and 17
# tiles (the latter among the chunks), 10 and 11 where the (KV head, sequence) pairs are no multiple of eight; up to 512 units with
# 18, 20 and 29 tiles; 516 and 528 units; rows of up to 4096 keys and longer ones.
POOLING_CASES = [
    (32, 8, 128, 1, 1, torch.float16, 1), (32, 8, 128, 33, 1, torch.bfloat16, 1), (32, 8, 128, 768, 1, torch.float16, 1),
    (28, 4, 128, 897, 1, torch.bfloat16, 0), (32, 8, 128, 843, 1, torch.float16, 1), (32, 8, 128, 1024, 1, torch.float16, 1),
    (32, 8, 64, 1024, 1, torch.float16, 1), (32, 8, 64, 1025, 1, torch.float16, 1), (8, 2, 64, 2049, 2, torch.bfloat16, 0),
    (40, 8, 128, 1050, 1, torch.float16, 1), (32, 8, 128, 1791, 1, torch.float16, 1), (28, 4, 128, 2081, 1, torch.float16, 0),
    (28, 4, 128, 2050, 1, torch.bfloat16, 0), (24, 8, 128, 1801, 1, torch.float16, 1), (14, 2, 64, 4128, 2, torch.float16, 1),
    (4, 4, 128, 4128, 1, torch.float16, 1), (4, 4, 128, 4129, 1, torch.float16, 0), (16, 1, 64, 517, 3, torch.float16, 1),
    (8, 2, 64, 1100, 3, torch.float16, 0), (14, 2, 128, 1300, 4, torch.bfloat16, 1), (36, 9, 64, 1281, 1, torch.float16, 1),
    (36, 9, 128, 1313, 1, torch.bfloat16, 0), (28, 4, 128, 1300, 2, torch.float16, 1), (28, 7, 64, 2300, 1, torch.float16, 1),
    (12, 3, 64, 2592, 2, torch.bfloat16, 1), (8, 2, 128, 3620, 2, torch.float16, 0), (12, 3, 64, 2800, 2, torch.float16, 1)]


def assert_pooling_route(G, D, B, q_start, rows, one_launch):
    from kascade_amd import _lib
    assert _lib.load().kascade_prefill_pool_selects(G, D, B, q_start, rows) == one_launch


@pytest.mark.parametrize("heads,G,D,L,B,dtype,one_launch", POOLING_CASES)
def test_pooling_that_selects_gives_the_lists_of_two_launches(cuda, heads, G, D, L, B, dtype, one_launch):
    """Prompts, strided and over shuffled pages: the lists of pooling and selection by calls of their own."""
    from kascade_amd import budgets, kernels
    assert_pooling_route(G, D, B, 0, L, one_launch)
    gen = torch.Generator().manual_seed(L + heads)
    q, k = _anchor_inputs(cuda, gen, heads, G, D, L, B, dtype)
    kp, table = _paged_copies(k[:1], 16, gen, 1, cuda)
    k = k.to(cuda)
    log_sum = kernels.prefill_recompute1(q, k)
    T = (L + 31) // 32
    for p, rolling in ((10, True), (5, False)):
        W = budgets.topk_width(L, p)
        valid, nsel = (torch.tensor(x, dtype=torch.int32, device=cuda)
                       for x in budgets.prefill_tile_budgets(L, 32, p, rolling, W))
        scores = torch.full((B, G, T, L), float("nan"), device=cuda, dtype=torch.float16)
        kernels.prefill_aggregate(q, k, log_sum, scores)
        want = kernels.topk_indices(scores, W, valid_len=valid, n_sel=nsel, fill_value=L - 1)
        got = kernels.prefill_anchor_topk(q, k, log_sum, torch.empty_like(scores), W, valid, nsel)
        assert torch.equal(got, want)
        own, rows = kernels.prefill_anchor_topk(q[:1], kp, log_sum[:1].contiguous(), torch.empty_like(scores[:1]), W, valid, nsel,
                                                block_table=table)
        assert torch.equal(own, want[:1]) and torch.equal(rows, kernels.translate_indices(own.contiguous(), table, L, 16))


POOLING_CHUNKS = [(32, 8, 128, 0, 512, 1, 1), (32, 8, 128, 1024, 1024, 1, 1), (32, 8, 128, 2048, 2048, 1, 1), (28, 4, 128, 2048, 2017, 1, 1),
                  (8, 2, 64, 256, 300, 4, 1), (64, 8, 128, 64, 500, 3, 1), (32, 8, 128, 800, 1280, 1, 1), (32, 8, 128, 832, 1280, 1, 0)]


@pytest.mark.parametrize("heads,G,D,start,n,B,one_launch", POOLING_CHUNKS)
def test_pooling_that_selects_over_chunks(cuda, heads, G, D, start, n, B, one_launch):
    """Chunks at one position and, with starts and row counts of their own (none and remainders among them), mixed ones:
    the lists and cache rows of two launches."""
    from kascade_amd import kernels
    assert_pooling_route(G, D, B, start, n, one_launch)
    from kascade_amd.strategy import PagedKascadePrefill
    gen = torch.Generator().manual_seed(start + n)
    L, T = start + n, (n + 31) // 32
    q, k = _anchor_inputs(cuda, gen, heads, G, D, L, B, torch.float16)
    kp, table = _paged_copies(k[:1], 8, gen, B, cuda)
    q = q[:, start:].contiguous()
    rule = PagedKascadePrefill(10, [list(range(G))], [0], page_size=8, device=cuda, kv_heads=G)
    starts = [(32 * b) % (start + 32) // 32 * 32 for b in range(B)]
    lens = [(n, 0, n - 17, 1)[b % 4] for b in range(B)]
    for mixed in (False, True):
        at, rows_of = (starts, lens) if mixed else (start, None)
        qs, qs_dev, ql_dev, s, c = rule._geometry(at, rows_of, n)
        Lk = qs + n
        W = 128 * -(-max(128, Lk // 10) // 128)
        valid, nsel = rule._ragged_budgets(s, c, n, W) if mixed else rule._tile_budgets(qs, n, W)
        log_sum, _ = kernels.prefill_chunk_dense(q, kp, kp, table, qs, 8, with_output=False, q_starts=qs_dev, q_lens=ql_dev)
        scores = torch.zeros(B, G, T, Lk, device=cuda, dtype=torch.float16)
        kernels.prefill_chunk_aggregate(q, kp, log_sum, scores, table, qs, 8, q_starts=qs_dev, q_lens=ql_dev)
        want = kernels.topk_indices(scores, W, valid_len=valid, n_sel=nsel, block_table=table, page_size=8)
        got = kernels.prefill_anchor_topk(q, kp, log_sum, torch.empty_like(scores), W, valid, nsel, block_table=table, q_start=qs,
                                          page_size=8, q_starts=qs_dev, q_lens=ql_dev)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), f"mixed {mixed}"


@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 60000.0])
def test_pooling_that_selects_takes_keys_of_every_value(cuda, value):
    """Keys that make scores infinite or no number, one and a whole tile of them: the lists of two launches."""
    from kascade_amd import budgets, kernels
    L, G = 700, 8
    assert_pooling_route(G, 128, 1, 0, L, 1)
    gen = torch.Generator().manual_seed(3)
    q, k = _anchor_inputs(cuda, gen, 32, G, 128, L, 1, torch.float16)
    k[0, 200:340, 1] = value
    k[0, 50, 2, 3] = value
    k = k.to(cuda)
    log_sum = kernels.prefill_recompute1(q, k)
    T, W = (L + 31) // 32, budgets.topk_width(L, 10)
    valid, nsel = (torch.tensor(x, dtype=torch.int32, device=cuda) for x in budgets.prefill_tile_budgets(L, 32, 10, True, W))
    scores = torch.empty(1, G, T, L, device=cuda, dtype=torch.float16)
    kernels.prefill_aggregate(q, k, log_sum, scores)
    want = kernels.topk_indices(scores, W, valid_len=valid, n_sel=nsel, fill_value=L - 1)
    assert torch.equal(kernels.prefill_anchor_topk(q, k, log_sum, torch.empty_like(scores), W, valid, nsel), want)


def test_pooling_that_selects_refuses_keys_of_other_sequences(cuda):
    """K of fewer sequences than Q, or of fewer positions, is refused before anything is launched."""
    from kascade_amd import kernels
    from kascade_amd._lib import KascadeError
    L, G = 64, 8
    q = torch.zeros(2, L, 32, 128, device=cuda, dtype=torch.float16)
    counts = torch.zeros(2, device=cuda, dtype=torch.int32)
    scores, log_sum = torch.zeros(2, G, 2, L, device=cuda, dtype=torch.float16), torch.zeros(2, L, 32, device=cuda)
    for k in (q[:1, :, :G], q[:, :L - 1, :G], torch.zeros(3, L, G, 128, device=cuda, dtype=torch.float16)):
        with pytest.raises(KascadeError, match="Q's sequences"):
            kernels.prefill_anchor_topk(q, k, log_sum, scores, 128, counts, counts)
    idx = kernels.prefill_anchor_topk(q, q[:1, :, :G].expand(2, -1, -1, -1), log_sum, scores, 128, counts, counts)
    assert idx.shape == (2, G, 2, 128) and bool((idx == L - 1).all())   # nothing selected: the filling


@pytest.mark.parametrize("heads,G,L,one_launch", [(32, 8, 700, 1), (28, 4, 897, 0)])
def test_pooling_that_selects_keeps_a_wrong_length_to_its_row(cuda, heads, G, L, one_launch):
    """A valid_len beyond the keys in front of its tile is the caller's mistake: that row's positions are unspecified below it,
    every other row's are as they were."""
    from kascade_amd import budgets, kernels
    assert_pooling_route(G, 128, 1, 0, L, one_launch)
    gen = torch.Generator().manual_seed(L)
    q, k = _anchor_inputs(cuda, gen, heads, G, 128, L, 1, torch.float16)
    k = k.to(cuda)
    log_sum = kernels.prefill_recompute1(q, k)
    T, W = (L + 31) // 32, budgets.topk_width(L, 10)
    valid, nsel = (torch.tensor(x, dtype=torch.int32, device=cuda) for x in budgets.prefill_tile_budgets(L, 32, 10, True, W))
    scores = torch.zeros(1, G, T, L, device=cuda, dtype=torch.float16)
    want = kernels.prefill_anchor_topk(q, k, log_sum, scores.clone(), W, valid, nsel)
    valid[T // 2] += 70
    got = kernels.prefill_anchor_topk(q, k, log_sum, scores, W, valid, nsel)
    rows = torch.arange(T, device=cuda) != T // 2
    assert torch.equal(got[:, :, rows], want[:, :, rows])
    taken = got[:, :, T // 2, :int(nsel[T // 2])]
    assert bool(((taken >= 0) & (taken < valid[T // 2])).all())


def _sparse_rows_as_documented(q, k, v, idx, p):
    """Rows of sparse units [L,H,D] with everything in 64 bits but the probabilities, which are rounded to the element type
    against references that the 32 queries of a block move together: when a score of any lies more than 2^8 above its own.
    Returns (these rows rounded to the element type, the rows in 64 bits, which rows belong to sparse units)."""
    from kascade_amd import budgets
    _, L, H, D = q.shape
    G, width, keys_per_tile = k.shape[2], idx.shape[-1], 64 * 128 // D
    gs = H // G
    rows, exact = (torch.zeros(L, H, D, dtype=torch.float64) for _ in range(2))
    sparse = torch.zeros(L, dtype=torch.bool)
    for t in range((L + 31) // 32):
        q0, end = 32 * t, min(32 * t + 32, L)
        n = min(budgets.rolling_budget(q0, p), width) if L > 128 else width
        if q0 <= n:
            continue
        sparse[q0:end] = True
        for g in range(G):
            listed = idx[0, g, t, :n].long()
            qq = q[0, q0:end, g * gs:(g + 1) * gs].double().transpose(0, 1)
            ref = torch.full((gs, end - q0, 1), -torch.inf, dtype=torch.float64)
            total, o, scores, values = torch.zeros_like(ref), 0.0, [], []
            for i, keys in enumerate([torch.arange(q0, end), *listed.split(keys_per_tile)]):
                s = qq @ k[0, keys, g].double().T * (D ** -0.5 / math.log(2))
                if i == 0:
                    s = s.masked_fill(torch.ones(end - q0, end - q0).triu(1).bool(), -torch.inf)
                scores.append(s)
                values.append(v[0, keys, g].double())
                top = s.amax(-1, keepdim=True)
                move = (top > ref + 8).any(1, keepdim=True)
                new = torch.where(move, torch.maximum(ref, top), ref)
                total, o, ref = total * torch.exp2(ref - new), o * torch.exp2(ref - new), new
                probs = torch.exp2(s - ref).to(q.dtype).double()
                total, o = total + probs.sum(-1, keepdim=True), o + probs @ values[-1]
            rows[q0:end, g * gs:(g + 1) * gs] = (o / total).to(q.dtype).double().transpose(0, 1)
            weights = torch.softmax(torch.cat(scores, -1) * math.log(2), -1)
            exact[q0:end, g * gs:(g + 1) * gs] = (weights @ torch.cat(values)).transpose(0, 1)
    return rows, exact, sparse


@pytest.mark.parametrize("heads,G,D,L,copies,dtype", [(8, 2, 128, 1100, 4, torch.float16), (8, 2, 64, 1100, 4, torch.bfloat16),
                                                      (7, 1, 128, 677, 7, torch.bfloat16)])
def test_sparse_rows_are_as_near_to_64_bits_as_their_references_allow(cuda, heads, G, D, L, copies, dtype):
    """Units in halves (one copy) and whole ones: the error against 64 bits is that of rounding the probabilities once, against
    references that move for a whole block.  Sums and products in 32 bits add less than 0.5 % to it; references that each
    query moved for its own scores alone added 2.4 to 5 %."""
    from kascade_amd import budgets, kernels
    p = 20
    gen = torch.Generator().manual_seed(L + D)
    q = (torch.randn(1, L, heads, D, generator=gen) * 3).to(dtype)
    k, v = (torch.randn(1, L, G, D, generator=gen).to(dtype) for _ in range(2))
    T, W = (L + 31) // 32, budgets.topk_width(L, p)
    idx = torch.zeros(1, G, T, W, dtype=torch.int32)
    for t in range(1, T):
        n = min(32 * t, W)
        for g in range(G):
            idx[0, g, t, :n] = torch.randperm(32 * t, generator=gen)[:n].sort().values
    rows, exact, sparse = _sparse_rows_as_documented(q, k, v, idx, p)
    least = (rows - exact)[sparse].norm()
    maps = torch.arange(G, dtype=torch.int32, device=cuda)
    for n in (1, copies):
        got = kernels.prefill_reuse(*(x.to(cuda).repeat(n, 1, 1, 1) for x in (q, k, v, idx)), maps, float(p), True)[-1]
        error = (got.cpu().double() - exact)[sparse].norm()
        assert float(error / least) <= 1.005, f"{n} copies: {float(error / exact[sparse].norm()):.4e}"
