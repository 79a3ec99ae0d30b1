"""The native page allocator (luc_blocks_*, lucciola-rs_amd/csrc/luc_blocks.cpp)
through the C ABI, on the CPU: the reference's single-sequence behaviour
(KVCache free list and prepare_for_step, src/layers/kv_cache.rs:73-76,
106-122), then a model-based check of many sequences against a plain Python
statement of the allocation rules."""
import dataclasses

import numpy as np
import pytest
import torch

from lucciola_rs_amd import model
from lucciola_rs_amd.engine import BlockManager
from lucciola_rs_amd.library import LucError

PAGE = 16


def test_single_sequence_matches_prepare_for_step():
    """Token by token, one sequence: the same pages as the reference's loop
    (pop from a free list filled in reverse when pos enters a new page)."""
    n = 40
    bm = BlockManager(n, 1, 64)
    free = list(range(n - 1, -1, -1))
    table = []
    for pos in range(300):
        if pos // PAGE >= len(table):
            table.append(free.pop())
        bm.reserve(0, pos + 1)
        row = bm.table()[0]
        assert list(row[: len(table)]) == table and not row[len(table):].any()
    assert bm.num_free == len(free) and bm.num_pages(0) == len(table)
    assert table == list(range(len(table)))  # a fresh pool hands out 0, 1, 2, ...


def test_multi_page_growth_and_no_shrink():
    bm = BlockManager(100, 2, 20)
    bm.reserve(0, 1)
    assert bm.num_pages(0) == 1
    bm.reserve(0, 5 * PAGE + 1)  # one call, five more pages
    assert bm.num_pages(0) == 6
    bm.reserve(0, 3)  # never shrinks
    assert bm.num_pages(0) == 6
    bm.reserve(1, 0)
    assert bm.num_pages(1) == 0


def test_out_of_pages_changes_nothing():
    bm = BlockManager(10, 3, 10)
    bm.reserve(0, 4 * PAGE)
    before = (bm.table().copy(), bm.num_free)
    with pytest.raises(LucError, match="LUC_E_NOMEM.*out of pages"):
        bm.reserve(1, 7 * PAGE)
    with pytest.raises(LucError, match="LUC_E_NOMEM"):
        bm.reserve_batch([1, 2], [3 * PAGE, 3 * PAGE + 1])  # 7 pages, 6 free: neither is given any
    assert np.array_equal(bm.table(), before[0]) and bm.num_free == before[1]
    bm.reserve_batch([1, 2], [3 * PAGE, 3 * PAGE])  # exactly the 6 free pages
    assert bm.num_free == 0


def test_invalid_arguments():
    bm = BlockManager(10, 2, 4)
    with pytest.raises(LucError, match="LUC_E_INVALID.*outside"):
        bm.reserve(2, 1)
    with pytest.raises(LucError, match="LUC_E_INVALID.*row holds 4"):
        bm.reserve(0, 4 * PAGE + 1)
    with pytest.raises(LucError, match="LUC_E_INVALID.*twice"):
        bm.reserve_batch([1, 1], [1, 1])
    with pytest.raises(LucError, match="LUC_E_INVALID.*negative"):
        bm.reserve(0, -1)
    with pytest.raises(LucError, match="LUC_E_INVALID"):
        bm.release(-1)
    with pytest.raises(LucError, match="LUC_E_INVALID"):
        BlockManager(0, 1, 1)
    assert bm.num_free == 10


def test_release_then_reserve_gives_the_same_pages():
    bm = BlockManager(64, 4, 16)
    bm.reserve(0, 50)
    bm.reserve(1, 100)
    row = bm.table()[1].copy()
    bm.release(1)
    bm.reserve(1, 100)
    assert np.array_equal(bm.table()[1], row)
    bm.release(3)  # releasing an empty sequence is a no-op
    assert bm.num_free == 64 - 4 - 7


class Model:
    """The allocation rules in plain Python."""

    def __init__(self, n, seqs, max_pages):
        self.free = list(range(n - 1, -1, -1))
        self.rows = [[] for _ in range(seqs)]
        self.max_pages = max_pages

    def reserve_batch(self, seqs, toks):
        extra = [max(0, -(-t // PAGE) - len(self.rows[s])) for s, t in zip(seqs, toks)]
        if any(-(-t // PAGE) > self.max_pages for t in toks):
            return "invalid"
        if sum(extra) > len(self.free):
            return "nomem"
        for s, e in zip(seqs, extra):
            for _ in range(e):
                self.rows[s].append(self.free.pop())
        return "ok"

    def release(self, s):
        self.free.extend(reversed(self.rows[s]))
        self.rows[s] = []


@pytest.mark.parametrize("seed", range(4))
def test_random_operations_against_the_rules(seed):
    rng = np.random.default_rng(seed)
    n, seqs, max_pages = 200, 12, 24
    bm, m = BlockManager(n, seqs, max_pages), Model(n, seqs, max_pages)
    for _ in range(600):
        op = rng.random()
        if op < 0.25:
            s = int(rng.integers(seqs))
            bm.release(s)
            m.release(s)
        else:
            k = int(rng.integers(1, 5))
            ss = rng.choice(seqs, size=k, replace=False).astype(np.int32)
            tt = rng.integers(0, max_pages * PAGE + 40, size=k).astype(np.int32)
            want = m.reserve_batch(list(ss), list(tt))
            try:
                bm.reserve_batch(ss, tt)
                got = "ok"
            except LucError as e:
                got = {-6: "nomem", -1: "invalid"}[e.code]
            assert got == want
        table = bm.table()
        for s in range(seqs):
            r = m.rows[s]
            assert list(table[s, : len(r)]) == r and not table[s, len(r):].any()
        assert bm.num_free == len(m.free)
        held = [p for r in m.rows for p in r]
        assert len(set(held)) == len(held) and len(held) + len(m.free) == n  # no page twice


class _NoLaunch:
    """Stands in for the library object: the model's host work runs, every
    launch is left out, and each attention call's block table is kept."""

    def __init__(self):
        self.tables = []
        self.lib = self

    def rope_table(self, max_pos, head_dim, base, scale):
        return torch.zeros(max_pos, head_dim // 2), torch.zeros(max_pos, head_dim // 2)

    def workspace_size(self, *a):
        return 0

    def luc_prompt_mlp_workspace_size(self, *a):
        return 0

    def decode_step(self, *a, **kw):
        self.tables.append(a[8].clone())

    def paged_prefill(self, *a, **kw):
        self.tables.append(a[8].clone())

    def __getattr__(self, name):
        return lambda *a, **kw: None


@pytest.mark.parametrize("calls", [
    [(40, 32)], [(100, 160)], [(5, 0), (20, 40)], [(64, 700)], [(1, 700)], [(2, 33)],
    [(33, 0), (1, 33), (1, 34)], [(16, 0), (16, 16), (1, 32), (40, 100)]])
def test_model_reserves_the_pages_of_every_position(calls):
    """Qwen2Model.forward at any start position, also past the reserved pages
    (a prefix loaded straight into the pools): when the attention runs, the
    table holds the pages 0, 1, 2, ... of every position up to the last row, none
    twice and none missing."""
    cfg = dataclasses.replace(model.QWEN25_05B, hidden_size=128, intermediate_size=128,
                              num_attention_heads=2, num_key_value_heads=1, num_hidden_layers=1,
                              vocab_size=64)
    lib = _NoLaunch()
    m = model.Qwen2Model(cfg, model.random_weights(cfg, 0), max_positions=1024, device="cpu", lib=lib)
    last = 0
    for rows, pos in calls:
        m.forward([1] * rows, pos)
        last = max(last, pos + rows)
        pages = -(-last // 16)
        assert m.kv.block_table_cpu == list(range(pages))
        assert lib.tables[-1].reshape(-1)[:pages].tolist() == list(range(pages))


@pytest.mark.parametrize("hidden,heads,kv,inter,kernels,library", [
    (256, 4, 2, 704, 6000, 30000), (512, 8, 2, 1408, 4096, 6000), (896, 14, 2, 4864, 700, 2500), (896, 14, 2, 4864, 1536, 4096), (1024, 16, 16, 2816, 1100, 2048),
    (1536, 12, 2, 8960, 700, 1281), (2048, 16, 2, 11008, 300, 769), (3584, 28, 4, 18944, 129, 700),
    (5120, 40, 8, 13824, 64, 257), (8192, 64, 8, 28672, 16, 200), (896, 14, 2, 4872, None, 5)])
def test_prompt_products_rule(hidden, heads, kv, inter, kernels, library):
    """Prompts run on the library GEMMs where these measured faster (large row
    counts and widths; sizes the kernels do not take), and on this library's own
    products elsewhere."""
    cfg = dataclasses.replace(model.QWEN25_05B, hidden_size=hidden, num_attention_heads=heads,
                              num_key_value_heads=kv, intermediate_size=inter)
    assert kernels is None or model.prompt_kernels_win(cfg, kernels)
    assert not model.prompt_kernels_win(cfg, library)


@pytest.mark.parametrize("rows,own", [(2, 1), (1536, 1), (1537, 0)])
def test_model_prompt_follows_the_rule(monkeypatch, rows, own):
    """Qwen2Model.forward launches luc_prompt_gemm once a layer where the rule
    says so, and not at all elsewhere."""
    cfg = dataclasses.replace(model.QWEN25_05B, hidden_size=128, intermediate_size=128,
                              num_attention_heads=2, num_key_value_heads=1, num_hidden_layers=2,
                              vocab_size=64)
    monkeypatch.setattr(model, "PROMPT_KERNEL_FEW", 0)
    lib = _NoLaunch()
    calls = []
    lib.prompt_gemm = lambda *a: calls.append(a[1].shape[0])
    m = model.Qwen2Model(cfg, model.random_weights(cfg, 0), max_positions=2048, device="cpu", lib=lib)
    m.forward([1] * rows, 0)
    assert calls == [rows] * 2 * own
