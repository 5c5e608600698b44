"""CPU tests of the host side: budgets, head-map loading, strategy construction and dispatch
arithmetic, synthetic workloads.  The oracle's closed forms are the reference values."""
import math

import pytest
import torch

from kascade_amd import budgets, workloads
from oracle import kascade_oracle as orc


@pytest.mark.parametrize("p", [5, 10, 20, 33, 12.5])
def test_budgets_match_oracle(p):
    for L in [129, 500, 2048, 4097, 16384, 32768, 65536, 131072, 524288]:
        assert budgets.topk_width(L, p) == orc.k_kern(L, p)
        assert budgets.decode_budget(L, p) == orc.n_kvcache(L, p)
    for ts in range(0, 40000, 32):
        assert budgets.rolling_budget(ts, p) == orc.n_kern(ts, p)


@pytest.mark.parametrize("rolling", [True, False])
def test_prefill_tile_budgets(rolling):
    L, tile, p = 5000, 32, 10
    K = budgets.topk_width(L, p)
    valid, nsel = budgets.prefill_tile_budgets(L, tile, p, rolling, K)
    T = math.ceil(L / tile)
    assert len(valid) == len(nsel) == T
    for t in range(T):
        assert valid[t] == t * tile
        assert nsel[t] == min(K, orc.prefill_budget(t, tile, L, p, rolling, K))
    # short prompts never roll (the reference switches rolling off for seq_len <= 128)
    v, n = budgets.prefill_tile_budgets(128, tile, p, True, 128)
    assert n == [128] * 4


def test_head_mapping_loader_and_strategy_ctor():
    from kascade_amd.strategy import EfficientKascadeStrategy, get_head_mapping
    from kascade_amd._lib import KascadeError
    hm = get_head_mapping("meta-llama/Meta-Llama-3.1-8B-Instruct", [0, 2, 8, 13, 14])
    assert len(hm) == 32 and all(len(r) == 8 for r in hm)
    for l in (0, 2, 8, 13, 14):
        assert hm[l] == list(range(8))
    hq = get_head_mapping("Qwen/Qwen3-8B", [0, 2, 7, 14, 23])
    assert len(hq) == 36
    with pytest.raises(ValueError):
        get_head_mapping("nobody/none", [0, 1])
    s = EfficientKascadeStrategy([0, 2, 8, 13, 14], "meta-llama/Meta-Llama-3.1-8B-Instruct", k=10, tile_size=32,
                                 rolling_prefill=True, register=False)
    assert s.name == "efficient_kascade" and s.k == 10 and s.tile_size == 32 and s.rolling_prefill
    assert s.recompute_layers == [0, 2, 8, 13, 14] and s._block_size == 12288
    assert s._head_mapping == hm and s._topk_to_reuse is None
    with pytest.raises(KascadeError):
        EfficientKascadeStrategy([0], None, k=10, tile_size=16, head_mapping=hm, register=False)
    with pytest.raises(KascadeError):
        EfficientKascadeStrategy([2], None, k=10, tile_size=32, head_mapping=hm, register=False)
    with pytest.raises(ValueError):
        EfficientKascadeStrategy([0], None, k=101, tile_size=32, head_mapping=hm, register=False)


def test_strategy_registers_with_hf():
    from transformers.modeling_utils import ALL_ATTENTION_FUNCTIONS
    from transformers.masking_utils import ALL_MASK_ATTENTION_FUNCTIONS
    from kascade_amd.strategy import EfficientKascadeStrategy
    hm = [list(range(8))] * 4
    s = EfficientKascadeStrategy([0], None, k=10, tile_size=32, head_mapping=hm, register=True)
    assert "efficient_kascade" in ALL_ATTENTION_FUNCTIONS.valid_keys()
    assert ALL_MASK_ATTENTION_FUNCTIONS["efficient_kascade"] is ALL_MASK_ATTENTION_FUNCTIONS["sdpa"]

    class M(torch.nn.Module):
        layer_idx = 0
        num_key_value_groups = 4
    # short contexts fall back to SDPA exactly like the reference (Lk <= 128), on any device
    q = torch.randn(1, 32, 16, 128)
    k = torch.randn(1, 8, 16, 128)
    v = torch.randn(1, 8, 16, 128)
    out, w = ALL_ATTENTION_FUNCTIONS["efficient_kascade"](M(), q, k, v, None, 128 ** -0.5, is_causal=True)
    ref = torch.nn.functional.scaled_dot_product_attention(
        q, k.repeat_interleave(4, 1), v.repeat_interleave(4, 1), is_causal=True).transpose(1, 2)
    assert w is None and torch.allclose(out, ref, atol=1e-5)


@pytest.mark.parametrize("Lk", [100, 128])
def test_short_context_falls_back_to_sdpa(Lk):
    """EfficientKascadeStrategy.py:137-140: up to 128 keys the call is SDPA with the caller's mask,
    prefill and decode alike, and the strategy's stored indices are not touched."""
    from kascade_amd.strategy import EfficientKascadeStrategy
    hm = [list(range(8))] * 2
    s = EfficientKascadeStrategy([0], None, k=10, tile_size=32, head_mapping=hm, register=False)

    class M(torch.nn.Module):
        layer_idx = 1
        num_key_value_groups = 4
    g = torch.Generator().manual_seed(Lk)
    k = torch.randn(2, 8, Lk, 128, generator=g)
    v = torch.randn(2, 8, Lk, 128, generator=g)
    for Lq in (Lk, 1):
        q = torch.randn(2, 32, Lq, 128, generator=g)
        mask = orc.causal_additive_mask(Lk, Lk, torch.float32)[:, :, Lk - Lq:]
        out, w = s.attention_forward(M(), q, k, v, mask.expand(2, 1, Lq, Lk), 128 ** -0.5)
        want, _ = orc.dense_prefill(torch.cat([torch.zeros(2, Lk - Lq, 32, 128), q.transpose(1, 2)], 1),
                                    k.transpose(1, 2), v.transpose(1, 2))
        assert w is None and tuple(out.shape) == (2, Lq, 32, 128)
        assert torch.allclose(out, want[:, Lk - Lq:], atol=2e-5)
    assert s._topk_to_reuse is None
    # one key more goes to the kernels, which need the HIP library and a GPU: no silent fallback
    from kascade_amd._lib import KascadeError
    k1 = torch.randn(2, 8, Lk + 29, 128, generator=g).half()
    q1 = torch.randn(2, 32, 1, 128, generator=g).half()
    with pytest.raises(KascadeError, match="before any anchor"):
        s.attention_forward(M(), q1, k1, k1, None, 128 ** -0.5)
    if not torch.cuda.is_available():
        M.layer_idx = 0
        with pytest.raises((KascadeError, RuntimeError)):
            s.attention_forward(M(), q1, k1, k1, None, 128 ** -0.5)


def test_default_num_split_heuristic(monkeypatch):
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    # config 2: 128 (sequence, head) pairs x 6656 rows -> ~512 workgroups
    assert kernels.default_num_split(128 * 6656, 6656) == 4
    # ragged config 3: splits sized by the total, the longest sequence gets the most
    ns = kernels.default_num_split(8 * 111616, 52480)
    rps = -(-52480 // ns)
    wgs = sum(-(-n // rps) for n in (13184, 19712, 26240, 52480)) * 8
    assert 400 <= wgs <= 640
    # launches too small to fill the device spread down to 128 rows per workgroup
    assert kernels.default_num_split(8 * 300, 300) == 2
    assert kernels.default_num_split(8 * 1664, 1664) == 13
    assert kernels.default_num_split(8 * 100, 100) == 1
    # gather launches: about 1664 rows per workgroup however large the total
    assert kernels.default_num_split(128 * 13184, 13184) == 4
    assert kernels.default_num_split(128 * 13184, 13184, cap_rows=kernels.GATHER_ROWS_PER_SPLIT) == 8
    assert kernels.default_num_split(128 * 6656, 6656, cap_rows=kernels.GATHER_ROWS_PER_SPLIT) == 4


def test_split_count_of_a_ragged_batch_with_known_lengths(monkeypatch):
    """With the lengths known, the non-empty workgroups are counted exactly: as many splits as
    fit two workgroups per compute unit, every sequence's count rounded up."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    cus = 256
    seq = [131072, 196608, 262144, 524288]

    def wgs(ns, rows, longest):
        rps = ((-(-longest // ns) + 63) // 64) * 64
        return 8 * sum(max(1, -(-n // rps)) for n in rows)

    ns = kernels.default_num_split(8 * sum(seq), max(seq), row_counts=seq)
    assert wgs(ns, seq, max(seq)) <= 2 * cus < wgs(ns + 1, seq, max(seq))
    rows = [budgets.decode_budget(n, 10) for n in seq]
    ns = kernels.default_num_split(8 * sum(rows), max(rows), cap_rows=kernels.GATHER_ROWS_PER_SPLIT, row_counts=rows)
    assert wgs(ns, rows, max(rows)) <= 2 * cus < wgs(ns + 1, rows, max(rows))
    # uniform batches: whole residencies, a second one once a split would pass ~4096 rows
    assert kernels.default_num_split(128 * 13184, 13184, cap_rows=kernels.GATHER_ROWS_PER_SPLIT,
                                     row_counts=[13184] * 16) == 4
    assert kernels.default_num_split(128 * 26240, 26240, cap_rows=kernels.GATHER_ROWS_PER_SPLIT,
                                     row_counts=[26240] * 16) == 8
    # a single sequence and launches too small to fill the device keep the plain rule
    assert kernels.default_num_split(8 * 1664, 1664, row_counts=[1664]) == 13
    assert kernels.default_num_split(8 * 600, 300, row_counts=[300, 300]) == kernels.default_num_split(8 * 600, 300)


@pytest.mark.parametrize("batch,heads,rows,want", [(8, 8, 3064, 4), (16, 8, 1564, 2), (2, 8, 9064, 16), (9, 8, 2564, 7), (12, 8, 1264, 5),
                                                   (36, 2, 5064, 7), (33, 8, 600, 1), (1, 8, 16384, 32), (4, 8, 3064, 8)])
def test_splits_of_equal_lists_fill_whole_rounds(monkeypatch, batch, heads, rows, want):
    """No count between one workgroup per compute unit and nearly two, with the lengths known or not; counts outside
    stay those of the nearest number of rows."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    lists = batch * heads
    assert kernels.default_num_split(lists * rows, rows, heads=heads) == want
    for hint in (None, [rows] * batch):
        for n in (rows, rows + 1, rows + 777, 3 * rows):
            ns = kernels.default_num_split(lists * n, n, heads=heads, row_counts=hint and [n] * batch)
            assert not 256 < lists * ns < 461 or lists > 256, (n, ns)


@pytest.mark.parametrize("lists,rows,cap,want", [(8, 40064, 0, 32), (8, 524352, 0, 32), (32, 131136, 0, 8), (64, 16448, 0, 4), (64, 32832, 0, 8), (8, 131136, 0, 32), (8, 134000, 0, 32), (4, 40064, 0, 64), (32, 16064, 0, 8),
                                                 (128, 3064, 0, 4), (8, 1664, 1664, 13), (8, 2176, 1664, 16), (8, 6144, 1664, 16),
                                                 (8, 6272, 1664, 32), (2, 12032, 1664, 64), (4, 11008, 1664, 64)])
def test_splits_of_few_lists(monkeypatch, lists, rows, cap, want):
    """Few streamed lists are one workgroup per compute unit, at any length measured up to 32 lists; small gathers stay within
    what their merge requests in one trip."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    assert kernels.default_num_split(lists * rows, rows, cap_rows=cap or None) == want


@pytest.mark.parametrize("rows,want", [(6656, {17: 3, 18: 3, 19: 3, 20: 3, 21: 3, 22: 4, 23: 4, 24: 4, 25: 2, 26: 2, 28: 2}),
                                       (13184, {17: 5, 18: 5, 19: 5, 20: 4, 21: 4, 22: 4, 23: 4, 24: 4, 25: 5, 26: 4, 28: 4})])
def test_gathers_of_equal_lists_counted_exactly(monkeypatch, rows, want):
    """As PagedKascadeDecoder plans the gathers of a batch with equal hints (17 lists of 6656 rows: 544 workgroups, two on
    every compute unit and a few more, 94.5 us, 408 88.2)."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    got = {n: kernels.default_num_split(8 * n * rows, rows, wgs_per_cu=1, cap_rows=kernels.GATHER_ROWS_PER_SPLIT,
                                        row_counts=[rows] * n, heads=8) for n in want}
    assert got == want


@pytest.mark.parametrize("batch,hint,room,dense,gather", [
    (1, 4096, 131072, 8, 2), (8, 3000, 131072, 2, 1), (8, 4096, 131072, 2, 2), (4, 8000, 131072, 8, 4), (2, 9000, 32768, 16, 8),
    (16, 1500, 32768, 2, 1), (16, 8192, 32768, 4, 2), (17, 8192, 32768, 3, 3), (26, 1024, 32768, 1, 1), (1, 32768, 131072, 32, 13),
    (1, 3000, 3064, 24, 1), (8, 3000, 3064, 4, 1), (16, 65536, 65600, 4, 2)])
def test_splits_of_hints_below_the_room(monkeypatch, batch, hint, room, dense, gather):
    """Equal hints of 1/4 and 1/32 of the room, and of all of it: the splits that each list has are those of lists of that
    length, as near as the limits on num_split and splits in steps of 64 rows come, not those of full ones."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())

    def splits(ns, rows, longest):
        return max(1, -(-rows // (((-(-longest // ns) + 63) // 64) * 64)))
    ns = kernels.default_num_split(8 * batch * hint, room, row_counts=[hint] * batch)
    assert splits(ns, hint, room) == dense
    rows, longest = budgets.decode_budget(hint, 10), budgets.decode_budget(room, 10)
    ns = kernels.default_num_split(8 * batch * rows, longest, wgs_per_cu=1, cap_rows=kernels.GATHER_ROWS_PER_SPLIT,
                                   row_counts=[rows] * batch, lone_rows=kernels.gather_lone_rows(4, 8 * batch))
    assert splits(ns, rows, longest) == gather


@pytest.mark.parametrize("total,want", [(8 * 65536, 64), (16 * 32768, 64), (8 * 65536 + 8, 64)])
def test_splits_of_a_batch_of_different_lengths(monkeypatch, total, want):
    """A total that happens to be a multiple of the longest list does not make the lists equal ones."""
    from kascade_amd import kernels, _lib

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    assert kernels.default_num_split(total, 65536, lengths="mixed") == want
    assert kernels.default_num_split(24 * 3064, 3064, lengths="mixed") == kernels.default_num_split(24 * 3064 + 1, 3064, lengths="mixed")


@pytest.mark.parametrize("batch,room,heads,group,dense,reuse", [
    (1, 131136, 8, 4, 64, 32), (1, 32832, 8, 4, 64, 26), (8, 3064, 8, 8, 4, 1), (8, 3564, 8, 4, 7, 1), (9, 2564, 8, 4, 7, 1),
    (4, 16064, 8, 4, 16, 8), (12, 8960, 8, 4, 5, 5), (8, 16448, 8, 4, 8, 4), (36, 5064, 2, 4, 7, 7)])
def test_splits_of_a_decoder_without_hints(monkeypatch, batch, room, heads, group, dense, reuse):
    """Its lists may be shorter than the room: no counts that pay for full ones alone (one round for few streamed lists, 16 splits
    of short gathers), and whole rounds only where they keep two thirds of the splits.  The gathers are planned as max_batch
    lists of max_topk, which is more than the budget of all tokens together."""
    from kascade_amd import _lib, kernels
    from kascade_amd.strategy import PagedKascadeDecoder

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    dec = PagedKascadeDecoder(10, [list(range(heads))], [0], batch, room, device="cpu", kv_heads=heads, group_size=group)
    assert (dec.ns_dense, dec.ns_reuse) == (dense, reuse)
    plans = []
    monkeypatch.setattr(kernels, "default_num_split", lambda *a, **k: plans.append((*a[:2], k["lengths"])) or 1)
    PagedKascadeDecoder(10, [list(range(heads))], [0], batch, room, device="cpu", kv_heads=heads, group_size=group)
    PagedKascadeDecoder(10, [list(range(heads))], [0], batch, room, device="cpu", kv_heads=heads, group_size=group,
                        total_tokens=batch * room // 2)
    assert plans[:2] == [(heads * batch * room, room, "capacity"), (heads * batch * dec.max_topk, dec.max_topk, "capacity")]
    assert [p[2] for p in plans[2:]] == ["mixed", "mixed"]


@pytest.mark.parametrize("batch,tokens,dense,anchor", [(26, 16384, 1, 1), (22, 32768, 1, 1), (16, 65536, 4, 8), (33, 32768, 1, 2), (8, 8192, 8, 8)])
def test_anchor_passes_take_twice_the_splits_of_two_rounds(monkeypatch, batch, tokens, dense, anchor):
    """Of more than 8192 rows, and only where there are two: one round of workgroups stays one."""
    from kascade_amd import _lib
    from kascade_amd.strategy import PagedKascadeDecoder

    class FakeLib:
        def kascade_device_cu_count(self):
            return 256
    monkeypatch.setattr(_lib, "init", lambda: FakeLib())
    dec = PagedKascadeDecoder(10, [list(range(8))], [0], batch, tokens + 64, device="cpu", seqlens_hint=[tokens] * batch)
    assert (dec.ns_dense, dec.ns_anchor) == (dense, anchor)


def test_workloads_are_seeded_and_shaped():
    a = workloads.prefill_inputs(1, 256, seed=3)
    b = workloads.prefill_inputs(1, 256, seed=3)
    assert torch.equal(a.q, b.q) and torch.equal(a.k, b.k) and a.head_mapping == b.head_mapping
    assert tuple(a.q.shape) == (1, 256, 32, 128) and tuple(a.k.shape) == (1, 256, 8, 128)
    assert a.q.dtype == torch.float16
    # reuse layer is correlated with the anchor (noise scale 0.3)
    d = (a.q_reuse.float() - a.q.float()).std()
    assert 0.25 < float(d) < 0.35
    # attention sink: token 0 scores high for every query
    s = torch.einsum("lhd,md->lhm", a.q[0, 128:].float(), a.k[0, :, 0].float())
    assert float((s[..., 0] > s[..., 1:].mean(-1)).float().mean()) > 0.95
    p = workloads.paged_decode_inputs([100, 37], seed=1)
    assert tuple(p.k_pages.shape) == (7 + 3, 16, 8, 128) and tuple(p.block_table.shape) == (2, 7)
    used = torch.cat([p.block_table[0, :7], p.block_table[1, :3]]).tolist()
    assert sorted(used) == list(range(10))
    kc = orc.paged_to_contiguous(p.k_pages, p.block_table, [100, 37])
    assert torch.equal(kc[1, 5], p.k_pages[p.block_table[1, 0], 5])


@pytest.mark.parametrize("group,limit", [(1, 384), (4, 384), (5, 512), (16, 512)])
def test_short_gather_lists_are_one_split(group, limit):
    from kascade_amd import kernels
    lone = kernels.gather_lone_rows(group)
    assert lone == limit
    # no device query below the limit; the general rule has the say above it
    assert kernels.default_num_split(8 * limit, limit, lone_rows=lone) == 1
    assert kernels.default_num_split(8 * 16 * 128, 128, row_counts=[128] * 16, lone_rows=lone) == 1


@pytest.mark.parametrize("group,lists,limit", [(1, 8, 256), (2, 63, 256), (2, 64, 384), (3, 1, 384), (4, 8, 384), (5, 8, 384),
                                               (7, 15, 384), (7, 16, 512), (8, 1, 512), (16, 8, 512)])
def test_lone_gather_split_depends_on_the_number_of_lists(group, lists, limit):
    """With few lists the workgroups of several splits find idle compute units: the groups whose merge is
    the cheaper part go to several splits earlier there."""
    from kascade_amd import kernels
    assert kernels.gather_lone_rows(group, lists) == limit


@pytest.mark.parametrize("where", ["subclass", "class", "instance"])
@pytest.mark.parametrize("Lq", [200, 1])
@pytest.mark.parametrize("layer", [0, 1])
def test_replaced_seams_are_called(monkeypatch, where, Lq, layer):
    """EfficientKascadeStrategy.py:72-123: each layer kind runs through a method of its own, and one put in its
    place -- in a subclass, on the class or on an instance that exists already -- gets the layer, with the
    reference's arguments ([B,L,heads,D] tensors, decode Q [B,H,D])."""
    from types import SimpleNamespace
    from kascade_amd.strategy import EfficientKascadeStrategy
    L, p = 200, 10
    name = {(200, 0): "_prefill_recomp_forward", (200, 1): "_prefill_reuse_forward",
            (1, 0): "_decode_recomp_forward", (1, 1): "_decode_reuse_forward"}[Lq, layer]
    seen = []

    def mine(self, Q, *rest):
        seen.append((self, Q, rest))
        return Q + 1
    kind = type("Mine", (EfficientKascadeStrategy,), {name: mine}) if where == "subclass" else EfficientKascadeStrategy
    s = kind([0], None, k=p, tile_size=32, head_mapping=[list(range(8))] * 2, register=False)
    if where == "class":
        monkeypatch.setattr(EfficientKascadeStrategy, name, mine)
    elif where == "instance":
        s.__dict__[name] = lambda Q, *rest: mine(s, Q, *rest)
    q = torch.randn(2, 32, Lq, 128).half()
    k, v = torch.randn(2, 8, L, 128).half(), torch.randn(2, 8, L, 128).half()
    o, none = s.attention_forward(SimpleNamespace(layer_idx=layer), q, k, v, None, 128 ** -0.5)
    assert none is None and len(seen) == 1
    who, Q, (K, V, *rest) = seen[0]
    assert who is s and torch.equal(o, q.transpose(1, 2) + 1)
    assert torch.equal(Q, q[:, :, 0] if Lq == 1 else q.transpose(1, 2))
    assert torch.equal(K, k.transpose(1, 2)) and torch.equal(V, v.transpose(1, 2))
    width = budgets.topk_width(L, p)
    assert rest == {(200, 0): [width, 32, 0, p], (200, 1): [p, 1], (1, 0): [width, 0], (1, 1): [1]}[Lq, layer]


def test_prefill_seam_refuses_tiles_the_kernels_do_not_have():
    """The reference's seam takes the tile size with each call; the kernels have one."""
    from kascade_amd._lib import KascadeError
    from kascade_amd.strategy import EfficientKascadeStrategy
    s = EfficientKascadeStrategy([0], None, k=10, tile_size=32, head_mapping=[list(range(8))], register=False)
    q, k = torch.zeros(1, 200, 32, 128).half(), torch.zeros(1, 200, 8, 128).half()
    for tile in (16, 64):
        with pytest.raises(KascadeError, match="tile_size"):
            s._prefill_recomp_forward(q, k, k, 128, tile, 0, 10)


@pytest.mark.parametrize("torch_here", [True, False])
@pytest.mark.parametrize("gxx_here", [True, False])
def test_library_builds_with_hipcc_alone(monkeypatch, tmp_path, torch_here, gxx_here):
    """The C library needs hipcc only; the extension module of the Python strategies needs torch, and any host
    compiler, ROCm's among them."""
    import shutil
    from pathlib import Path
    from kascade_amd import build
    ran = []

    def run(cmd):
        ran.append([str(x) for x in cmd])
        Path(ran[-1][ran[-1].index("-o") + 1]).touch()
        return ""
    monkeypatch.setattr(build, "_run", run)
    monkeypatch.setattr(build, "PKG_DIR", tmp_path)
    monkeypatch.setattr(build, "LIB_PATH", tmp_path / "libkascade_hip.so")
    monkeypatch.setattr(build, "NATIVE_PATH", tmp_path / "_native.so")
    monkeypatch.setattr(build, "_hipcc", lambda: "/opt/rocm/bin/hipcc")
    if not torch_here:
        monkeypatch.setattr(build, "_torch_root", lambda: None)
    which = shutil.which
    monkeypatch.setattr(shutil, "which", lambda name: (which(name) if gxx_here or name != "g++" else None))
    assert build.build() == tmp_path / "libkascade_hip.so" and build.LIB_PATH.exists()
    native = [c for c in ran if any("native.cpp" in x for x in c)]
    assert len(native) == (1 if torch_here else 0) and build.NATIVE_PATH.exists() == torch_here
    assert all(c[0] == "/opt/rocm/bin/hipcc" for c in ran if c not in native)
    if native and not gxx_here:
        assert native[0][0].endswith("amdclang++")
    count = len(ran)
    build.ensure_built()
    assert len(ran) == count
