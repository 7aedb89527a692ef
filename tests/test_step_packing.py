"""The host side of the step function (no GPU): the integers that a step hands to the kernels, for
random mixed traces over the cache manager.  Every token's cache row must be the one its block
table names, sequences of one token come first, wanted rows follow the entries' order, and the
rows that pad a step to a fixed shape own nothing."""
import numpy as np
import pytest

import helpers
from deliverance_amd.cache.manager import CacheManager, KVGroupSpec, StateSpec
from deliverance_amd.engine.step import StepEntry, StepPacker
from deliverance_amd.sampling.sampler import RECORD_WORDS


def pack(packer, mgr, entries, pad_to=None, max_blocks=None, extra=None):
    starts = {}
    for e in entries:
        if e.rid not in mgr:
            mgr.open(e.rid)
        starts[e.rid] = mgr.extend(e.rid, len(e.tokens))
    order = sorted(range(len(entries)), key=lambda i: (len(entries[i].tokens) != 1, i))
    offs, meta, n_words = packer.layout(entries, order, pad_to=pad_to, max_blocks=max_blocks, extra=extra)
    buf = np.full(n_words, -12345, dtype=np.int32)
    packer.fill(buf, offs, meta, entries, order, starts, extra)
    assert not (buf == -12345).any(), "a word of the step was left unwritten"
    return order, starts, meta, {k: buf[a:a + n] for k, (a, n) in offs.items()}


@pytest.mark.parametrize("seed,page,groups", [(0, 16, 1), (1, 32, 2), (2, 64, 1), (3, 16, 2)])
def test_mixed_traces_pack_consistently(seed, page, groups):
    rng = np.random.default_rng(seed)
    P, V = 333, 1000
    lengths = [int(x) for x in rng.integers(1, P - 1, size=6)] + [P - 1]
    reqs = [(f"r{i}", [int(t) for t in rng.integers(0, V, size=n)]) for i, n in enumerate(lengths)]
    steps = helpers.trace_mixed(reqs, seed=seed, prefill_sizes=(9, 2, 67, 4, 130, 33), decode_tail=int(rng.integers(1, 20)))
    n_pages = helpers.max_live_tokens(steps, round_to=max(64, page)) // page
    specs = [KVGroupSpec((2 * g, 2 * g + 1), 2, 16, None) for g in range(groups)]
    mgr = CacheManager(specs, page, [n_pages] * groups, [StateSpec(9, 4)], 4)
    packer = StepPacker(mgr, groups, page)
    given = {rid: 0 for rid, _ in reqs}
    ids = dict(reqs)
    for st in steps:
        entries = [StepEntry(e["id"], e["tokens"], e["want"]) for e in st["entries"]]
        if entries:
            order, starts, meta, v = pack(packer, mgr, entries)
            N, S, mb = meta["N"], meta["S"], meta["max_blocks"]
            assert N == sum(len(e.tokens) for e in entries) and S == len(entries)
            # one-token sequences first, each kind in the entries' order
            kinds = [len(entries[i].tokens) != 1 for i in order]
            assert kinds == sorted(kinds) and meta["n_decode"] == kinds.count(False)
            qs, sl = v["q_start"], v["seq_lens"]
            assert qs[0] == 0 and qs[-1] == N and (np.diff(qs) > 0).all()
            for s, i in enumerate(order):
                e = entries[i]
                rows = slice(int(qs[s]), int(qs[s + 1]))
                assert v["tokens"][rows].tolist() == list(e.tokens) == ids[e.rid][given[e.rid]:given[e.rid] + len(e.tokens)]
                assert v["positions"][rows].tolist() == list(range(given[e.rid], given[e.rid] + len(e.tokens)))
                assert (v["seq_of"][rows] == s).all() and (v["token_src"][rows] == -1).all()
                assert sl[s] == given[e.rid] + len(e.tokens)
                assert v["state_slots"][s] == mgr.state_slot(e.rid) >= 0
                for g in range(groups):
                    bt = v[f"block_table{g}"].reshape(S, mb)
                    table = mgr.table(e.rid, g)
                    assert bt[s, :len(table)].tolist() == table and (bt[s, len(table):] == -1).all()
                    assert len(table) == -(-int(sl[s]) // page) and all(0 <= p < n_pages for p in table)
                    for row, pos in zip(range(rows.start, rows.stop), v["positions"][rows]):
                        assert v[f"slot_map{g}"][row] == table[pos // page] * page + pos % page
            for g in range(groups):
                assert len(set(v[f"slot_map{g}"].tolist())) == N          # no cache row is written twice
            # wanted rows: in the order of the entries (not of the sequences) and of each entry's `want`
            first_row = {i: int(qs[s]) for s, i in enumerate(order)}
            assert v["want"].tolist() == [first_row[i] + w for i, e in enumerate(entries) for w in e.want]
            for e in entries:
                mgr.commit(e.rid)
                given[e.rid] += len(e.tokens)
        for rid in st["end"]:
            mgr.close(rid)
        mgr.check()
    assert all(pool.n_free == n_pages for pool in mgr.pools)


def test_padding_rows_own_nothing():
    """A decode step padded to a fixed shape: the added sequences have length 0, no cache row, no
    state, and their sampling records are zero."""
    page, n_pages = 16, 32
    mgr = CacheManager([KVGroupSpec((0,), 2, 16, None)], page, [n_pages])
    packer = StepPacker(mgr, 1, page)
    for rid, n in (("a", 20), ("b", 3), ("c", 40)):
        mgr.open(rid)
        mgr.extend(rid, n)
        mgr.commit(rid)
    entries = [StepEntry(rid, [7], [0]) for rid in ("a", "b", "c")]
    extra = list(range(1, 3 * RECORD_WORDS + 1))
    order, starts, meta, v = pack(packer, mgr, entries, pad_to=8, max_blocks=64, extra=extra)
    assert meta["S"] == meta["N"] == meta["R"] == 8 and meta["n_decode"] == 8 and meta["max_blocks"] == 64
    assert v["seq_lens"].tolist() == [21, 4, 41, 0, 0, 0, 0, 0]
    assert v["positions"].tolist() == [20, 3, 40, 0, 0, 0, 0, 0]
    assert (v["slot_map0"][3:] == -1).all() and (v["slot_map0"][:3] >= 0).all()
    assert (v["state_slots"] == -1).all()                 # this manager keeps no state
    assert (v["block_table0"].reshape(8, 64)[3:] == -1).all()
    assert v["want"].tolist() == list(range(8))
    assert v["extra"][:len(extra)].tolist() == extra and (v["extra"][len(extra):] == 0).all()
    assert len(v["extra"]) == 8 * RECORD_WORDS


def test_a_single_token_may_come_from_the_step_before():
    mgr = CacheManager([KVGroupSpec((0,), 1, 16, None)], 16, [8])
    packer = StepPacker(mgr, 1, 16)
    mgr.open("a"); mgr.extend("a", 5); mgr.commit("a")
    order, starts, meta, v = pack(packer, mgr, [StepEntry("a", [0], [0], from_sampled=3), StepEntry("b", [4, 5, 6], [2])])
    assert v["token_src"].tolist() == [3, -1, -1, -1] and v["positions"].tolist() == [5, 0, 1, 2]


def test_a_launch_that_fails_leaves_no_reservation_behind(tmp_path):
    """The step function reserves positions, then launches.  When the launch is refused (here: the
    kernels are asked to run on CPU tensors, which they refuse) the reservation goes back and the
    requests that the call opened are closed; a request that was open before keeps what it had."""
    import torch
    import helpers
    from deliverance_amd.engine.device_cache import DeviceCache
    from deliverance_amd.engine.step import StepEntry
    from deliverance_amd.kernels import ops
    from deliverance_amd.models.causal_lm import load_model
    from simt import harness
    m = helpers.make_model(tmp_path, helpers.CONFIG_A, 0)
    model = load_model(m.folder, torch.float32, "cpu")
    with pytest.raises(ValueError, match="page_size must be one of"):
        DeviceCache(model.cache_needs(), torch.float32, "cpu", 48, 256, n_state_slots=4)
    cache = DeviceCache(model.cache_needs(), torch.float32, "cpu", 16, 256, n_state_slots=4)
    runner = harness.make_runner(model, cache)          # the step function without pinned memory
    mgr = cache.manager
    mgr.open("old")
    mgr.extend("old", 20)
    mgr.commit("old")
    free = mgr.pools[0].n_free
    with pytest.raises((ops.KernelError, RuntimeError)):       # no GPU here: the first launch refuses
        runner.run([StepEntry("old", [1] * 30, [29]), StepEntry("new", [2] * 40, [])])
    assert mgr.live() == ["old"] and mgr.length("old") == 20 and mgr.pending("old") == 0
    assert mgr.pools[0].n_free == free
    mgr.check()


def arena_bytes(arena, name):
    held = [t for key, t in arena._bufs.items() if key[0] == name] + [e[0] for key, e in arena._flats.items() if key[0] == name]
    return len(held), sum(t.numel() * t.element_size() for t in held)


def native_step(monkeypatch, tmp_path, **rules):
    """The plan of a step issued from C++, without a library behind it, and a context of a step of N rows on an arena."""
    import torch
    from types import SimpleNamespace
    from deliverance_amd.engine.device_cache import DeviceCache
    from deliverance_amd.engine.native_step import NativeStep
    from deliverance_amd.kernels import ops
    from deliverance_amd.models.causal_lm import load_model
    from deliverance_amd.parts.base import Arena, StepContext
    monkeypatch.setattr(ops, "_lib", lambda: SimpleNamespace(da_run_step=lambda *a: 0, da_attn_both_pays=lambda *a: 0))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    for name, rule in rules.items():
        monkeypatch.setattr(ops, name, rule)
    model = load_model(helpers.make_model(tmp_path, helpers.CONFIG_A, 0).folder, torch.bfloat16, "cpu")
    cache = DeviceCache(model.cache_needs(), torch.bfloat16, "cpu", 16, 256, n_state_slots=4)
    arena = Arena("cpu")

    def context(N, n_decode, blocks):
        ctx = StepContext()
        ctx.n_tokens, ctx.n_seqs, ctx.n_decode, ctx.max_query_len = N, max(1, n_decode), n_decode, 1 if n_decode else N
        ctx.tokens = ctx.positions = ctx.seq_of_token = ctx.q_start = ctx.seq_lens = torch.zeros(N + 1, dtype=torch.int32)
        ctx.block_tables, ctx.slot_maps, ctx._arena = [torch.zeros(ctx.n_seqs, blocks, dtype=torch.int32)], [ctx.tokens], arena
        return ctx
    return NativeStep(model, cache), arena, context


def test_scratch_of_steps_of_many_sizes_is_one_buffer(monkeypatch, tmp_path):
    """The plan of a step issued from C++ asks for scratch whose size follows the step's: over steps of many sizes, in no
    order, an engine keeps one buffer of each kind, at most twice the largest need, and a size within the largest one
    allocates nothing."""
    shares = lambda M, N, K: max(1, min(8, 2048 // M)) if M > 8 else 1
    step, arena, context = native_step(monkeypatch, tmp_path, step_shares=shares)
    width = step.model.config.width
    largest = 0
    for N in [int(n) for n in np.random.default_rng(3).permutation(np.arange(1, 1500, 7))]:
        before = arena_bytes(arena, "proj_partial")
        step.forward(context(N, 0, 4), None, 0)
        need = 4 * shares(N, width, 0) * N * width if shares(N, width, 0) > 1 else 0
        if need <= largest:
            assert arena_bytes(arena, "proj_partial") == before
        largest = max(largest, need)
        assert step._step.proj_partial_floats * 4 == need
    count, held = arena_bytes(arena, "proj_partial")
    assert count == 1 and largest <= held <= 2 * largest


@pytest.mark.parametrize("native", [True, False])
def test_scratch_of_decode_attention_of_many_sizes_is_one_buffer(monkeypatch, tmp_path, native):
    """Likewise the partial results of decode attention that shares a pair's keys out, in steps issued either way."""
    import torch
    from deliverance_amd.kernels import ops
    splits = lambda n_seqs, n_heads, blocks, page: max(1, min(blocks // 4, 512 // (n_seqs * n_heads)))
    step, arena, context = native_step(monkeypatch, tmp_path, decode_splits=splits, step_shares=lambda *a: 1,
                                       attention_decode=lambda *a, **k: None)
    at = step.model.blocks[0].mixer
    cache_slot = step.cache.kv[0]
    largest = 0
    for n, blocks in [(int(i) // 8 + 1, int(i) % 8 * 16 + 8) for i in np.random.default_rng(5).permutation(240)]:
        ctx = context(n, n, blocks)
        if native:
            step.forward(ctx, None, 0)
        else:
            q = torch.zeros(n, at.n_heads * at.head_dim, dtype=torch.bfloat16)
            with ops.kernel_mode_scope("tuned"):
                ops.paged_attention(ctx, q, cache_slot, 0, at.n_heads, 1.0, None, torch.empty_like(q))
        k = splits(n, at.n_heads, blocks, 16)
        if k > 1:
            largest = max(largest, 4 * ops.decode_workspace_floats(n, at.n_heads, at.head_dim, k))
    count, held = arena_bytes(arena, "decode_partial")
    assert count == 1 and 0 < largest <= held <= 2 * largest


@pytest.mark.parametrize("joins", [False, True])
def test_parts_share_products_out_only_where_norms_add_the_shares(monkeypatch, joins):
    """A feed-forward's second product adds into the stream in one kernel, unless the model's steps are issued from C++, whose
    norms add the shares in passing: any other model would pay for a kernel of its own."""
    import torch
    from types import SimpleNamespace
    from deliverance_amd.kernels import ops
    from deliverance_amd.parts.base import Arena, StepContext
    from deliverance_amd.parts.feedforward import DenseFeedForward
    calls = []
    for name in ("linear", "linear_shares", "join_rows"):
        monkeypatch.setattr(ops, name, lambda *a, _n=name, **k: calls.append(_n))
    monkeypatch.setattr(ops, "shares_ok", lambda *a: True)
    monkeypatch.setattr(ops, "step_shares", lambda M, N, K: 4)
    monkeypatch.setattr(ops, "product_shares", lambda M, N, K: 4, raising=False)
    ff = DenseFeedForward(SimpleNamespace(width=16, inner=64, activation="gelu_new", bias=False),
                          {"fc_weight": torch.zeros(64, 16), "proj_weight": torch.zeros(16, 64)}, torch.bfloat16, "cpu")
    ctx = StepContext()
    ctx._arena, ctx.dtype = Arena("cpu"), torch.bfloat16
    if joins:
        ctx.joins_shares = True
    ff.forward(ctx, torch.zeros(100, 16, dtype=torch.bfloat16), torch.zeros(100, 16))
    assert calls == (["linear", "linear_shares", "join_rows"] if joins else ["linear", "linear"])
