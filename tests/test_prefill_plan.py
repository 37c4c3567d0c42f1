"""Host-side tile tables of chunked prefill: the fused kernel's query tiles and
the two-pass path's workspace and query tiles cover every query row and every
context key exactly once (echokv_vllm/kernels/prefill.py:56-87)."""

import numpy as np

from echokv_amd.kernels import prefill as pf


def test_tiles_cover_every_query_row():
    prefill = [(0, 70, 70, 0), (70, 110, 200, 0), (110, 111, 33, 0)]
    for gqa in (1, 4, 7):
        tiles = pf.build_tiles(prefill, [0, 1, 2], gqa, "cpu")
        covered = sorted(r for q0, n, *_ in tiles.tolist() for r in range(q0, q0 + n))
        assert covered == list(range(111))
        assert all(n <= pf.block_m(gqa) for _, n, *_ in tiles.tolist())
        assert tiles[0].tolist()[2] == 0 and any(x[2] == 160 for x in tiles.tolist())


def test_dense_plan_covers_rows_and_contexts():
    prefill = [(0, 70, 70, 0), (70, 110, 200, 0), (110, 111, 33, 0), (111, 611, 900, 0)]
    for gqa in (1, 4, 7):
        plan = pf.build_dense_plan(prefill, [0, 1, 2, 5], gqa, "cpu")
        qt, packs = plan.qtiles.tolist(), plan.packs.tolist()
        covered = sorted(r for q0, n, *_ in qt for r in range(q0, q0 + n))
        assert covered == list(range(611))
        assert all(0 < n <= pf.dense_block_m(gqa) for _, n, *_ in qt)
        for q0, n, pos0, ctx, t0 in qt:
            (qs, qe, c, _), r = next((p, r) for p, r in zip(prefill, [0, 1, 2, 5]) if p[0] <= q0 < p[1])
            assert ctx == c and pos0 == c - (qe - qs) + (q0 - qs)
            keys = [k0 for rr, k0, cc in packs[t0 : t0 + -(-c // pf.DENSE_KEYS)]]
            assert keys == list(range(0, c, pf.DENSE_KEYS))
            assert all(rr == r and cc == c for rr, _, cc in packs[t0 : t0 + len(keys)])
        # heaviest request first
        assert qt[0][3] == 900


def test_fused_prefill_refuses_tiles_larger_than_its_kernel_takes():
    """Tiles built for the MFMA kernel (block_m tokens) handed to a layout that
    takes the fp32 kernel (any_block_m tokens) are refused on the host, tagged
    or not, before any device work; tiles of the right size pass the check."""
    import pytest
    import torch
    from types import SimpleNamespace

    store = SimpleNamespace(layout=SimpleNamespace(num_kv_heads=2, head_size=80), pages=torch.zeros(1))
    gqa = 4
    q = torch.zeros(40, 2 * gqa, 80)
    prefill, req = [(0, 40, 40, 0)], [0]
    assert not pf.kernels_take(80, gqa) and pf.block_m(gqa) > pf.any_block_m(gqa)
    big = pf.build_tiles(prefill, req, gqa, "cpu")
    for tiles in (big, big.clone()):  # tagged by build_tiles, and an untagged copy
        with pytest.raises(ValueError, match="at most"):
            pf.prefill_attention_fused(store, q, q, prefill, req, torch.zeros(1, 1), 0.1, tiles)
    ok = pf.build_tiles(prefill, req, gqa, "cpu", tokens=pf.any_block_m(gqa))
    with pytest.raises(RuntimeError, match="device tensors"):  # past the check: CPU tensors are refused next
        pf.prefill_attention_fused(store, q, q, prefill, req, torch.zeros(1, 1), 0.1, ok)


def test_head_size_256_tiles_hold_half_the_rows():
    """At head size 256 the fused MFMA kernel takes 64 query rows per tile (64 //
    GQA tokens): tiles built at head size 128's size are refused on the host,
    tiles of the right size pass; own-group-exact prefill is not offered there."""
    import pytest
    import torch
    from types import SimpleNamespace

    gqa = 4
    assert pf.kernels_take(256, gqa) and not pf.own_group_takes(256, gqa) and pf.own_group_takes(128, gqa)
    assert pf.block_m(gqa, 256) == 16 and pf.block_m(gqa) == 32 and not pf.kernels_take(256, 80)
    store = SimpleNamespace(layout=SimpleNamespace(num_kv_heads=2, head_size=256), pages=torch.zeros(1))
    q = torch.zeros(40, 2 * gqa, 256)
    prefill, req = [(0, 40, 40, 0)], [0]
    with pytest.raises(ValueError, match="at most"):
        pf.prefill_attention_fused(store, q, q, prefill, req, torch.zeros(1, 1), 0.1,
                                   pf.build_tiles(prefill, req, gqa, "cpu"))
    ok = pf.build_tiles(prefill, req, gqa, "cpu", tokens=pf.block_m(gqa, 256))
    with pytest.raises(RuntimeError, match="device tensors"):
        pf.prefill_attention_fused(store, q, q, prefill, req, torch.zeros(1, 1), 0.1, ok)
    with pytest.raises(ValueError, match="own-group"):
        pf.prefill_attention(store, q, q, prefill, req, torch.zeros(1, 1), 0.1, own_group_key=q)


def test_fused_key_ranges_come_from_the_request_alone():
    """A request's range length: 256 or 512 keys or more, whole steps of every head size's
    kernel, at most 64 ranges a tile, and over 512 keys at most 64 of the request's tiles
    unless a tile is one range; the same in any batch."""
    for tiles in (1, 2, 3, 7, 32, 64, 500):
        for ctx in (1, 511, 512, 513, 4096, 32767, 32768, 32769, 65537, 200000, 1 << 20):
            per = pf.range_keys(tiles, ctx)
            assert per >= 256 and per % 128 == 0 and -(-ctx // per) <= pf.MAX_RANGES
            assert ctx > pf.ONE_RANGE or ctx <= per
            assert per > 256 or tiles * -(-ctx // per) <= pf.FEW_RANGES
            assert tiles * -(-ctx // per) <= pf.MANY_RANGES or ctx <= per
    one = (0, 40, 3000, 0)
    other = [(40, 41, 100, 0), (41, 105, 30000, 0)]
    alone = pf.build_tiles([one], [0], 4, "cpu").ranges.host_items
    among = pf.build_tiles([one, *other], [0, 1, 2], 4, "cpu").ranges.host_items
    assert (among[: len(alone), [0, 1, 2, 4]] == alone[:, [0, 1, 2, 4]]).all()


def test_fused_range_plan_covers_every_tile_within_its_rows():
    """Every tile's keys are covered once by its items, in order; its partial rows are its own
    within its group, and a group's fit the limit unless it is one tile. The largest
    step's partial rows stay within PARTIAL_BYTES: 60 chunks of 64 tokens beside one over 32K keys
    took 1.0 GB when every query row had room for the most ranges."""
    rng = np.random.default_rng(5)
    steps = [[(0, 64, 8192, 0)], [(0, 1, 1, 0)], [(64 * i, 64 * i + 64, 64 if i else 32768, 0) for i in range(61)],
             [(512 * i, 512 * i + 512, 4096, 0) for i in range(16)], [(0, 3, 200000, 0), (3, 10, 513, 0)],
             [(40 * i, 40 * i + int(rng.integers(1, 40)), int(rng.integers(40, 5000)), 0) for i in range(50)]]
    for prefill in steps:
        for gqa, heads, d in ((4, 8, 128), (8, 1, 128), (1, 32, 64), (4, 8, 256)):
            tiles = pf.build_tiles(prefill, list(range(len(prefill))), gqa, "cpu", tokens=pf.block_m(gqa, d))
            plan = tiles.ranges
            items, merges = plan.items.view(-1, 5).tolist(), plan.merges.view(-1, 5).tolist()
            want = []
            for t, (_, n, p0, ctx, req) in enumerate(tiles.tolist()):
                per, keys = pf.range_keys(int((tiles[:, 4] == req).sum()), ctx), min(p0 + n, ctx)
                want += [(t, z, -(-keys // per), per, n * gqa) for z in range(-(-keys // per))]
            assert [(i // 64, i % 64, n, per, r) for i, n, per, _, r in items] == want
            assert merges == [it for it in items if it[0] % 64 == 0 and it[1] > 1]
            for limit in (1, 1000, pf.PARTIAL_BYTES // (heads * (d + 2) * 4)):
                g, most = plan.groups(limit)
                assert [sum(x[1] for x in g[:i]) for i in range(len(g) + 1)] == [x[0] for x in g] + [len(items)]
                assert [sum(x[3] for x in g[:i]) for i in range(len(g) + 1)] == [x[2] for x in g] + [len(merges)]
                for i0, n, m0, nm, row0 in g:
                    used, at = 0, row0
                    assert merges[m0 : m0 + nm] == [it for it in items[i0 : i0 + n] if it[0] % 64 == 0 and it[1] > 1]
                    for _, ranges, _, first, rows in merges[m0 : m0 + nm]:
                        assert first == at
                        at += ranges * rows
                    used = at - row0
                    assert used <= most and (used <= limit or nm == 1)
            if len(prefill) > 2:
                assert most * heads * (d + 2) * 4 <= pf.PARTIAL_BYTES


def test_fused_prefill_plans_its_ranges_once(monkeypatch):
    """A table from build_tiles carries its ranges: a layer's call plans nothing."""
    import pytest
    import torch
    from types import SimpleNamespace

    store = SimpleNamespace(layout=SimpleNamespace(num_kv_heads=2, head_size=128), pages=torch.zeros(1))
    prefill = [(0, 40, 4000, 0)]
    tiles = pf.build_tiles(prefill, [0], 4, "cpu")

    def plan(*_):
        raise AssertionError("planned again")

    monkeypatch.setattr(pf, "RangePlan", plan)
    monkeypatch.setattr(pf._lib, "require_device", lambda *_: None)
    q = torch.zeros(40, 8, 128)
    with pytest.raises(AttributeError, match="res_k"):  # past the planning, at the store's buffers
        pf.prefill_attention_fused(store, q, q, prefill, [0], torch.zeros(1, 1, dtype=torch.int32), 0.1, tiles)
