"""The Qwen2 decoder loop on the HIP path (lucciola_rs_amd/model.py) against
the oracle's restatement (oracle/model.py): the model loop's small kernels
bit for bit, and a random-init Qwen2.5-0.5B (24 layers, hidden 896, 14q/2kv,
intermediate 4864, vocab 151936, tied embeddings) generating greedily for 128
steps after a prefill."""
import numpy as np
import pytest
import torch

from lucciola_rs_amd import model as model_module
from lucciola_rs_amd.model import QWEN25_05B, Qwen2Config, Qwen2Model, random_weights, to_bf16_bits
from gpu_util import from_dev, say, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _needs_device():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")


def bf16_ulps(a, b):
    """Distance in bf16 units in the last place between two bit arrays (finite values)."""
    def key(x):
        x = x.astype(np.int32)
        return np.where(x & 0x8000, -(x & 0x7fff), x & 0x7fff)
    return np.abs(key(a) - key(b))


def test_rmsnorm_bit_exact(orc, luc):
    rng = np.random.default_rng(1)
    for rows, cols in [(1, 896), (7, 896), (3, 4864), (2, 64), (5, 2056), (1, 8192), (2, 8200)]:
        x = to_bf16_bits(rng.standard_normal((rows, cols)) * rng.uniform(0.1, 30))
        w = to_bf16_bits(1 + 0.1 * rng.standard_normal(cols))
        want = orc.rmsnorm(x, w, 1e-6)
        tx, tw = to_dev(x, "bf16"), to_dev(w, "bf16")
        out = torch.empty_like(tx)
        say(f"  [gpu] rmsnorm rows={rows} cols={cols}")
        luc.rmsnorm(out, tx, tw, 1e-6)
        luc.rmsnorm(tx, tx, tw, 1e-6)  # in place
        torch.cuda.synchronize()
        assert np.array_equal(from_dev(out), want)
        assert np.array_equal(from_dev(tx), want)


def test_silu_mul_matches_oracle(orc, luc):
    """f32 silu * up rounded to bf16; the GPU's expf and the host's may differ
    in the last f32 bit, so a bf16 result may rarely differ by one unit."""
    rng = np.random.default_rng(2)
    rows, inter = 9, 4864
    gu = to_bf16_bits(rng.standard_normal((rows, 2 * inter)) * 3)
    want = orc.silu_mul(gu.copy(), inter)
    t = to_dev(gu, "bf16")
    say(f"  [gpu] silu_mul rows={rows} inter={inter}")
    luc.silu_mul(t, inter)
    torch.cuda.synchronize()
    got = from_dev(t)
    assert np.array_equal(got[:, inter:], gu[:, inter:])  # up untouched
    d = bf16_ulps(got[:, :inter], want[:, :inter])
    say(f"  max ulp {d.max()}, differing {np.count_nonzero(d)} of {d.size}")
    assert d.max() <= 1 and np.count_nonzero(d) <= d.size // 1000


@pytest.mark.parametrize("n,k,res", [
    (1152, 896, False),    # q/k/v of Qwen2.5-0.5B
    (896, 896, True),      # o, residual add in place
    (9728, 896, False),    # gate | up
    (896, 4864, True),     # down, residual add in place
    (1001, 1024, False),   # rows not a multiple of 16, the widest four-row k
    (37, 1032, True),      # the narrowest one-row k, rows not a multiple of 4
    (5, 8192, False),      # the widest k
    (3, 8, True),          # the narrowest k
])
def test_gemv_against_f64(luc, n, k, res):
    """y = x w^T (+ residual) for one bf16 row (models.rs:252-295 at M = 1):
    f32 products summed in a fixed order, one rounding to bf16.  Against the
    f64 sum rounded once, an f32 sum of k <= 8192 terms can differ only where
    the exact result lies within ~k * 2^-24 (relative) of a bf16 rounding
    boundary: at most one unit, and rarely."""
    rng = np.random.default_rng(n * 31 + k)
    x = to_bf16_bits(rng.standard_normal(k))
    w = to_bf16_bits(rng.standard_normal((n, k)) * 0.05)
    r = to_bf16_bits(rng.standard_normal(n) * 4) if res else None
    f = lambda b: (b.astype(np.uint32) << 16).view(np.float32).astype(np.float64)  # noqa: E731
    exact = f(w) @ f(x) + (f(r) if res else 0.0)
    want = to_bf16_bits(exact.astype(np.float32))  # f64 -> f32 -> bf16: off by one unit at worst
    tx, tw = to_dev(x, "bf16"), to_dev(w, "bf16")
    y = to_dev(r, "bf16") if res else torch.empty(n, dtype=torch.bfloat16, device="cuda")
    say(f"  [gpu] gemv n={n} k={k} residual={res}")
    luc.gemv(y, tx, tw, residual=y if res else None)
    torch.cuda.synchronize()
    d = bf16_ulps(from_dev(y), want)
    say(f"  max ulp {d.max()}, differing {np.count_nonzero(d)} of {d.size}")
    assert d.max() <= 1 and np.count_nonzero(d) <= max(2, d.size // 100)


@pytest.mark.parametrize("n,k,res", [
    (1152, 896, False), (9728, 896, True), (37, 4864, False), (5, 8192, True), (3, 8, False),
    (4096, 1024, False), (7, 1032, True),
    (65537, 896, True), (70001, 1024, False),   # eight rows a wave (lm_head's shape class)
])
def test_rmsnorm_gemv_equals_unfused(luc, n, k, res):
    """luc_rmsnorm_gemv forms RMSNorm(x) in each wave with luc_rmsnorm's
    arithmetic order, so it must give luc_rmsnorm then luc_gemv bit for bit."""
    rng = np.random.default_rng(n * 7 + k)
    x = to_bf16_bits(rng.standard_normal(k) * rng.uniform(0.1, 30))
    nw = to_bf16_bits(1 + 0.1 * rng.standard_normal(k))
    w = to_bf16_bits(rng.standard_normal((n, k)) * 0.05)
    r = to_bf16_bits(rng.standard_normal(n)) if res else np.zeros(n, np.uint16)
    tx, tn, tw = to_dev(x, "bf16"), to_dev(nw, "bf16"), to_dev(w, "bf16")
    y1, y2 = to_dev(r, "bf16"), to_dev(r, "bf16")
    norm = torch.empty_like(tx)
    say(f"  [gpu] rmsnorm_gemv n={n} k={k} residual={res}")
    luc.rmsnorm(norm, tx, tn, 1e-6)
    luc.gemv(y1, norm, tw, residual=y1 if res else None)
    luc.rmsnorm_gemv(y2, tx, tn, 1e-6, tw, residual=y2 if res else None)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(y1), from_dev(y2))


@pytest.mark.parametrize("inter,k,norm", [
    (4864, 896, True),     # Qwen2.5-0.5B's gate/up
    (4864, 896, False), (1001, 1024, True), (3, 8, True), (37, 1032, False), (5, 8192, True),
    (8960, 1536, True),    # Qwen2.5-1.5B's gate/up
    (11, 5128, False),     # the narrowest k of the sixteen-chunk pair
])
def test_gate_up_silu_equals_unfused(luc, inter, k, norm):
    """luc_gate_up_silu rounds each gate and up product to bf16 and applies
    luc_silu_mul's arithmetic to the pair, so it must give luc_rmsnorm (or
    nothing), luc_gemv into [gate | up] and luc_silu_mul bit for bit.  (The
    unfused pair runs on gate and up padded to a multiple of 8 rows, which
    luc_silu_mul needs.)"""
    rng = np.random.default_rng(inter * 3 + k)
    x = to_bf16_bits(rng.standard_normal(k) * rng.uniform(0.1, 30))
    nw = to_bf16_bits(1 + 0.1 * rng.standard_normal(k))
    pad = -(-inter // 8) * 8
    w = to_bf16_bits(rng.standard_normal((2, pad, k)) * (2.0 / np.sqrt(k)))
    tx, tn = to_dev(x, "bf16"), to_dev(nw, "bf16")
    tw, tw_pad = to_dev(w[:, :inter].reshape(2 * inter, k), "bf16"), to_dev(w.reshape(2 * pad, k), "bf16")
    dev = dict(dtype=torch.bfloat16, device="cuda")
    say(f"  [gpu] gate_up_silu inter={inter} k={k} norm={norm}")
    xn = torch.empty_like(tx)
    if norm:
        luc.rmsnorm(xn, tx, tn, 1e-6)
    else:
        xn.copy_(tx)
    gu = torch.empty(2 * pad, **dev)
    luc.gemv(gu, xn, tw_pad)
    luc.silu_mul(gu, pad)
    act = torch.full((inter,), float("nan"), **dev)
    luc.gate_up_silu(act, tx, tn if norm else None, 1e-6, tw)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(act), from_dev(gu[:inter]))


@pytest.mark.parametrize("n,k", [
    (67, 512), (67, 520), (2047, 1024), (67, 1536), (67, 1544), (2049, 2048), (513, 2056),
    (4099, 2560), (67, 3072), (67, 3080), (67, 4096), (67, 4104), (67, 5120), (67, 5128),
    (67, 6144), (1537, 6152), (67, 6152), (2049, 6152), (3073, 6152)])
def test_one_row_products_at_variant_edges(luc, n, k):
    """Every chunk count and row count of the dispatch, at the edges of its k
    range and with n not a multiple of the rows a workgroup takes: the plain
    product against f64, the fused ones against the unfused, bit for bit."""
    test_gemv_against_f64(luc, n, k, True)
    test_rmsnorm_gemv_equals_unfused(luc, n, k, False)
    test_gate_up_silu_equals_unfused(luc, n, k, True)


def test_gemv_rejects_bad_shapes(luc):
    """k outside [8, 8192] or not a multiple of 8, and mismatched operands,
    are refused before any launch."""
    from lucciola_rs_amd.library import LucError
    dev = dict(dtype=torch.bfloat16, device="cuda")
    for k in (12, 8200, 0):
        w = torch.zeros(4, k, **dev)
        with pytest.raises(LucError):
            luc.gemv(torch.empty(4, **dev), torch.zeros(k, **dev), w)
    with pytest.raises(ValueError):
        luc.gemv(torch.empty(5, **dev), torch.zeros(64, **dev), torch.zeros(4, 64, **dev))
    with pytest.raises(ValueError):
        luc.gemv(torch.empty(4, **dev), torch.zeros(72, **dev), torch.zeros(4, 64, **dev))


def test_embedding_gather_and_out_of_range(luc):
    rng = np.random.default_rng(3)
    vocab, hidden = 1000, 896
    table = to_bf16_bits(rng.standard_normal((vocab, hidden)))
    ids = np.array([0, 999, 5, 5, 1000, 123], np.int32)  # 1000 is past the table
    out = torch.empty(len(ids), hidden, dtype=torch.bfloat16, device="cuda")
    say("  [gpu] embedding")
    luc.embedding(out, to_dev(table, "bf16"), torch.from_numpy(ids).cuda())
    torch.cuda.synchronize()
    got = from_dev(out)
    for r, i in enumerate(ids):
        if i < vocab:
            assert np.array_equal(got[r], table[i])
        else:
            assert np.all((got[r] & 0x7fff) > 0x7f80)  # NaN row


def test_argmax_ties_nan_and_floor(orc, luc):
    """luc_argmax against the oracle and the stated tie order of the
    reference's kernel (smallest i mod 1024, then smallest i): random rows,
    equal maxima (600 and 1500: 1500 wins), a NaN, nothing above -1e30."""
    import pins
    rng = np.random.default_rng(4)
    idx = torch.zeros(1, dtype=torch.int32, device="cuda")
    for c in pins.argmax_cases(rng):
        want = pins.argmax_tie_order(orc.to_f32(c, "bf16"))
        assert orc.argmax(c) == want
        # the row at the start of its buffer and one element in
        padded = to_dev(np.concatenate([np.zeros(1, np.uint16), c]), "bf16")
        for row in (to_dev(c, "bf16"), padded[1:]):
            say(f"  [gpu] argmax n={c.size} offset={(row.data_ptr() % 16) // 2}")
            idx.fill_(-7)
            luc.argmax(row, idx)
            torch.cuda.synchronize()
            assert int(idx.cpu().item()) == want


@pytest.fixture(scope="module")
def qwen():
    """Random-init Qwen2.5-0.5B (seeded; HF-style init: N(0, 0.02^2) matrices
    and biases, norm weights about 1) on the GPU and in the oracle."""
    from oracle.model import OracleQwen2
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    cfg = QWEN25_05B
    say("  building random-init Qwen2.5-0.5B weights")
    w = random_weights(cfg, seed=2025)
    max_pos = 512
    return cfg, Qwen2Model(cfg, w, max_positions=max_pos), OracleQwen2(cfg, w, max_pos)


class OracleAttentionModel(Qwen2Model):
    """The same GPU model with its attention (RoPE, cache write, attention)
    computed by the oracle: the layer's qkv rows go to the host, the oracle's
    restatement of the reference (orc_decode_step / orc_prefill: rope.cu,
    kv_cache.cu, attention.cu) runs on a host copy of the paged cache, and
    its output comes back.  Every other step -- embedding, RMSNorm, the
    GEMMs, silu * up, the logits GEMM, argmax -- is the GPU model's own, so
    two such models differ in attention only."""

    def __init__(self, orc, *a, **kw):
        super().__init__(*a, **kw)
        self.orc = orc
        self.k_host = np.zeros(tuple(self.kv.k_pool.shape), np.uint16)
        self.v_host = np.zeros(tuple(self.kv.v_pool.shape), np.uint16)
        self.cos_host = self.rope.cos.cpu().numpy()
        self.sin_host = self.rope.sin.cpu().numpy()
        self.bias_host = [tuple(from_dev(L[k]) for k in ("q_bias", "k_bias", "v_bias"))
                          for L in self.layers]

    def _oracle(self, li, qkv, run, first_pos):
        cfg = self.cfg
        qb, kb, vb = self.bias_host[li]
        table = self.kv.block_table.view(1, -1).cpu().numpy().astype(np.int32)
        rows = from_dev(qkv).copy()
        att = run(rows, (qb, kb, vb, self.cos_host, self.sin_host, self.k_host, self.v_host, table),
                  li, cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim,
                  float(np.float32(1.0) / np.sqrt(np.float32(cfg.head_dim))), 16,
                  cfg.num_hidden_layers, "bf16")
        att = self._finish(li, rows, table[0], first_pos, att)
        return to_dev(att.reshape(rows.shape[0], -1), "bf16")

    def _finish(self, li, roped_rows, table, first_pos, att):
        """The attention output of the layer (bits), given the oracle's."""
        return att

    def _attention_decode(self, li, qkv, pos):
        return self._oracle(li, qkv, lambda rows, args, *rest: self.orc.decode_step(
            rows, *args, np.array([pos], np.int32), *rest), pos)

    def _attention_prefill(self, li, qkv, cache_pos, cu, start):
        S = qkv.shape[0]
        return self._oracle(li, qkv, lambda rows, args, *rest: self.orc.prefill(
            rows, *args, np.array([0, S], np.int32), np.array([cache_pos], np.int32), *rest),
            cache_pos)


class ExactAttentionModel(OracleAttentionModel):
    """The oracle-attention model with the attention itself done in f64 and
    rounded once to bf16: textbook softmax(q K^T * scale) V over the same
    roped q and the same cache (both written by the oracle, bit-exact with
    the reference's rope.cu / kv_cache.cu), every other step the GPU
    model's.  It measures how far the reference's own f32 algorithm
    (attention.cu: 32 interleaved partitions, expf, one merge) lands from
    exact arithmetic, which bounds what any attention can be expected to
    reproduce through 24 layers of bf16 rounding."""

    def _finish(self, li, roped_rows, table, first_pos, att):
        cfg, orc = self.cfg, self.orc
        hq, hkv, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
        S = roped_rows.shape[0]
        pos = first_pos + np.arange(S)
        ctx = int(pos[-1]) + 1
        npg = (ctx + 15) // 16
        f64 = lambda b: orc.to_f32(b, "bf16").astype(np.float64)  # noqa: E731
        K = f64(self.k_host[table[:npg], li]).transpose(1, 0, 2, 3).reshape(hkv, npg * 16, d)[:, :ctx]
        V = f64(self.v_host[table[:npg], li]).transpose(1, 0, 2, 3).reshape(hkv, npg * 16, d)[:, :ctx]
        q = f64(roped_rows[:, : hq * d]).reshape(S, hq, d)
        scale = float(np.float32(1.0) / np.sqrt(np.float32(d)))
        late = np.arange(ctx)[None, :] > pos[:, None]
        out = np.empty((S, hq, d))
        G = hq // hkv
        for h in range(hq):
            sc = q[:, h] @ K[h // G].T * scale
            sc[late] = -np.inf
            p = np.exp(sc - sc.max(axis=1, keepdims=True))
            out[:, h] = (p @ V[h // G]) / p.sum(axis=1, keepdims=True)
        return to_bf16_bits(out.reshape(S, hq * d))


# Top-2 logit gap at or below which a greedy step counts as a near-tie that
# rounding may decide either way: 4 bf16 units at the logits' magnitude
# (2..4).  Any two attentions that differ in the last f32 bit of one output
# round one bf16 output differently now and then, and 24 layers of bf16
# rounding amplify that to 0.04-0.07 in the logits -- exact f64 attention
# against the reference's f32 algorithm included (measured: 0.049 after a
# 128-token prompt).
ATTN_LOGIT_NOISE = 0.0625


def greedy_compare(orc, models, prompt, steps=128):
    """Prefill `prompt`, then `steps` greedy steps, every model fed the first
    model's (the oracle attention's) greedy token each step (EOS/BOS stop
    bypassed, as models.rs:218, :236 would stop both alike).  For every other
    model: tokens that agree with the first's, the first step where they
    differ (the free-running prefix: up to it both ran on their own tokens),
    the worst logit difference against the first, and the steps where the
    first's top-2 gap exceeds ATTN_LOGIT_NOISE (decided) and whether those
    agree."""
    ref = models[0]
    n = len(models) - 1
    st = [dict(agree=0, prefix=None, worst=0.0, decided=0, decided_differ=[], differ=[])
          for _ in range(n)]
    ids, pos = prompt, 0
    for step in range(steps + 1):
        for m in models:
            m.forward(ids, pos)
        rl = orc.to_f32(from_dev(ref.logits())[0], "bf16")
        r = ref.sample_greedy()
        top2 = np.sort(rl)[-2:]
        gap = float(top2[1] - top2[0])
        for k, m in enumerate(models[1:]):
            ml = orc.to_f32(from_dev(m.logits())[0], "bf16")
            diff = float(np.max(np.abs(ml - rl)))
            g = m.sample_greedy()
            s = st[k]
            s["worst"] = max(s["worst"], diff)
            if gap > ATTN_LOGIT_NOISE:
                s["decided"] += 1
            if g == r:
                s["agree"] += 1
            else:
                s["prefix"] = step if s["prefix"] is None else s["prefix"]
                s["differ"].append((step, round(gap, 4), round(diff, 4)))
                if gap > ATTN_LOGIT_NOISE:
                    s["decided_differ"].append(step)
        pos += len(ids)
        ids = [r]
    for s in st:
        s["prefix"] = steps + 1 if s["prefix"] is None else s["prefix"]
        s["exempt"] = steps + 1 - s["decided"]
    return st


def report(name, s, steps):
    say(f"  {name}: {s['agree']} of {steps + 1} tokens identical, free-running prefix "
        f"{s['prefix']}; {s['decided']} decided steps (oracle top-2 gap > {ATTN_LOGIT_NOISE}), "
        f"{len(s['decided_differ'])} of them differ; {s['exempt']} near-tie steps exempt; "
        f"worst logit difference {s['worst']:.4f} ({s['worst'] / ATTN_LOGIT_NOISE:.0%} of the "
        f"bound); differing steps (step, gap, diff): {s['differ'][:12]}")


def test_greedy_128_steps_attention_swapped(orc):
    """The 128-step greedy check with attention as the only difference:
    random-init Qwen2.5-0.5B, a 128-token prompt, then 128 greedy steps
    (models.rs:195-240, greedy dispatch :398-405), three times with identical
    GPU GEMMs -- with the oracle's attention (OracleAttentionModel, the
    reference's algorithm), with this library's (luc_paged_prefill for the
    prompt, luc_decode_step per token) and with f64 textbook attention over
    the oracle's cache (ExactAttentionModel) -- each step fed the oracle
    run's token, so every step compares the attentions on the same history.
    Asserted for the library's attention: every decided step (oracle top-2
    gap above ATTN_LOGIT_NOISE) identical, at most 13 differing tokens, and a
    worst logit difference within twice the one exact arithmetic shows
    against the reference's algorithm.  The free-running prefix, the exempt
    near-tie steps and the headroom are reported for both: measured, exact
    arithmetic leaves the reference's greedy path at step 2 (119 of 129
    tokens identical), this library's attention at step 16 (124 of 129)."""
    cfg = QWEN25_05B
    w = random_weights(cfg, seed=2025)
    max_pos = 512
    ref = OracleAttentionModel(orc, cfg, w, max_positions=max_pos)
    hip = Qwen2Model(cfg, w, max_positions=max_pos)
    exact = ExactAttentionModel(orc, cfg, w, max_positions=max_pos)
    rng = np.random.default_rng(29)
    prompt = rng.integers(0, cfg.vocab_size, 128).tolist()
    say("  [gpu] prefill 128 + 128 greedy steps: oracle attention vs HIP attention vs f64 attention")
    sh, se = greedy_compare(orc, [ref, hip, exact], prompt)
    report("HIP attention vs oracle attention", sh, 128)
    report("f64 attention vs oracle attention", se, 128)
    assert not sh["decided_differ"], "a decided step differs"
    assert sh["worst"] <= 2 * max(se["worst"], 1 / 64)
    assert 129 - sh["agree"] <= 13


def test_greedy_after_2048_token_prefill(orc):
    """The prefill configuration's follow-on: random-init Qwen2.5-0.5B, the
    first of the 4 x 2048 seeded prompts (token ids uniform over the 151936
    vocab) through luc_paged_prefill in one call per layer, then 128 greedy
    steps with luc_decode_step, against the same model with the oracle's
    attention (its prefill restates the reference's per-token loop,
    models.rs:485-550, on the host), and with f64 textbook attention
    (ExactAttentionModel), each step fed the oracle run's token.  Every
    decided step must be identical, at most 13 tokens may differ, and the
    worst logit difference must stay within twice the one exact arithmetic
    shows against the reference's algorithm; the free-running prefix and the
    exempt near-tie steps are reported for both."""
    cfg = QWEN25_05B
    w = random_weights(cfg, seed=2025)
    max_pos = 2048 + 160
    ref = OracleAttentionModel(orc, cfg, w, max_positions=max_pos)
    hip = Qwen2Model(cfg, w, max_positions=max_pos)
    exact = ExactAttentionModel(orc, cfg, w, max_positions=max_pos)
    prompt = np.random.default_rng(2048).integers(0, cfg.vocab_size, (4, 2048))[0].tolist()
    say("  [gpu] prefill 2048 (luc_paged_prefill vs the oracle's per-token loop vs f64) + 128 greedy steps")
    sh, se = greedy_compare(orc, [ref, hip, exact], prompt)
    report("HIP attention vs oracle attention after 2048 prompt tokens", sh, 128)
    report("f64 attention vs oracle attention after 2048 prompt tokens", se, 128)
    assert not sh["decided_differ"], "a decided step differs"
    assert sh["worst"] <= 2 * max(se["worst"], 1 / 64)
    assert 129 - sh["agree"] <= 13


def test_greedy_lockstep_full_oracle(orc, qwen):
    """End to end against the oracle's whole loop (oracle/model.py, its GEMMs
    on the host BLAS): a 32-token prompt, then 128 steps teacher-forced by the
    oracle's greedy token.  The GEMMs' summation orders differ
    (luc_prompt_gemm here, BLAS in the oracle, cuBLAS in the reference), so where the two
    greedy tokens differ the step must be a near-tie: the GPU's token within
    that step's largest logit difference of the oracle's best.  At least 90%
    of the steps must agree."""
    cfg, gpu, ref = qwen
    rng = np.random.default_rng(17)
    prompt = rng.integers(0, cfg.vocab_size, 32).tolist()
    say("  [gpu] prefill 32 + 128 steps (GPU model and full oracle, teacher-forced by the oracle)")
    ids, pos, agree = prompt, 0, 0
    for step in range(129):
        gpu.forward(ids, pos)
        ref.forward(ids, pos)
        g, r = gpu.sample_greedy(), ref.sample_greedy()
        if g != r:
            gl = orc.to_f32(from_dev(gpu.logits())[0], "bf16")
            rl = orc.to_f32(ref.logits(), "bf16")
            diff = float(np.max(np.abs(gl - rl)))
            say(f"  step {step}: GPU {g} vs oracle {r}; oracle logits {rl[g]:.4f} vs {rl[r]:.4f}, "
                f"max |logit diff| {diff:.4f}")
            assert rl[r] - rl[g] <= diff, "a decided step differs"
        else:
            agree += 1
        pos += len(ids)
        ids = [r]
    say(f"  {agree} of 129 steps agree")
    assert agree >= 116


def test_teacher_forced_logits_random_tokens(orc, qwen):
    """Both loops fed the same seeded random tokens (after a fresh 16-token
    prefill at position 0 of a second cache): logits agree to within a few bf16
    units, and the argmax agrees wherever the oracle's top two logits are
    apart by more than the largest logit difference seen."""
    cfg, _, _ = qwen
    from oracle.model import OracleQwen2
    w = random_weights(cfg, seed=2025)
    gpu, ref = Qwen2Model(cfg, w, max_positions=256), OracleQwen2(cfg, w, 256)
    rng = np.random.default_rng(23)
    toks = rng.integers(0, cfg.vocab_size, 16 + 48).tolist()
    say("  [gpu] teacher-forced: prefill 16, then 48 random tokens")
    worst, flips, decided = 0.0, 0, 0
    for step in range(49):
        ids, pos = (toks[:16], 0) if step == 0 else ([toks[15 + step]], 15 + step)
        gpu.forward(ids, pos)
        ref.forward(ids, pos)
        gl = orc.to_f32(from_dev(gpu.logits())[0], "bf16")
        rl = orc.to_f32(ref.logits(), "bf16")
        diff = float(np.max(np.abs(gl - rl)))
        worst = max(worst, diff)
        top2 = np.sort(rl)[-2:]
        if top2[1] - top2[0] > 2 * diff:
            decided += 1
            flips += int(np.argmax(gl) != np.argmax(rl))
    say(f"  max |logit diff| {worst:.4f}; argmax compared on {decided} of 49 steps, {flips} differ")
    assert worst < 0.1
    assert flips == 0


@pytest.mark.parametrize("inter", [512, 8200])
def test_greedy_from_checkpoint_second_shape(orc, tmp_path, inter):
    """A written-then-loaded checkpoint at another head shape (hidden 256, 4q/2kv,
    3 layers, vocab 1000, untied lm_head, rope scaling 2): the GPU loop and the
    oracle in lockstep for a 20-token prompt and 48 greedy steps, with the same
    near-tie rule as above.  Intermediate 8200 takes the down projection of a
    decode step past the GEMV's 8192 onto a GEMM."""
    from oracle.model import OracleQwen2
    from lucciola_rs_amd.checkpoint import load_checkpoint, write_checkpoint
    from lucciola_rs_amd.model import Qwen2Config
    cfg = Qwen2Config(vocab_size=1000, hidden_size=256, num_hidden_layers=3, num_attention_heads=4,
                      num_key_value_heads=2, intermediate_size=inter, max_position_embeddings=4096,
                      tie_word_embeddings=False, rope_scaling_factor=2.0, eos_token_id=999,
                      bos_token_id=998)
    write_checkpoint(str(tmp_path), cfg, random_weights(cfg, seed=31, std=0.08), shards=2)
    gpu = Qwen2Model.from_checkpoint(str(tmp_path), max_positions=128)
    cfg2, w2 = load_checkpoint(str(tmp_path))
    ref = OracleQwen2(cfg2, w2, 128)
    ids = np.random.default_rng(19).integers(0, cfg.vocab_size, 20).tolist()
    pos, tokens = 0, []
    say("  [gpu] checkpoint model: prefill 20 + 48 greedy steps in lockstep")
    for step in range(49):
        gpu.forward(ids, pos)
        ref.forward(ids, pos)
        g, r = gpu.sample_greedy(), ref.sample_greedy()
        if g != r:
            gl = orc.to_f32(from_dev(gpu.logits())[0], "bf16")
            rl = orc.to_f32(ref.logits(), "bf16")
            diff = float(np.max(np.abs(gl - rl)))
            say(f"  step {step}: GPU {g} vs oracle {r}; {rl[g]:.4f} vs {rl[r]:.4f}, diff {diff:.4f}")
            assert rl[r] - rl[g] <= diff
            break
        tokens.append(g)
        pos += len(ids)
        ids = [g]
    say(f"  identical for {len(tokens)} of 49 tokens; distinct: {len(set(tokens))}")
    assert len(tokens) >= 24


def test_sample_token_dispatch(orc, qwen):
    """Qwen2Model.sample_token (models.rs:385-432) on the model's own logits:
    temperature 0 is luc_argmax; top_p < 1 draws, with the sampler's first
    random value, the token the oracle's apply_sort_and_sample draws from the
    same logits (checked where no interval end lies within 1e-5 of top_p or
    the target; always among the oracle's candidates)."""
    import pins
    from lucciola_rs_amd.sampler import Sampler
    cfg, gpu, _ = qwen
    rng = np.random.default_rng(23)
    gpu.forward(rng.integers(0, cfg.vocab_size, 5).tolist(), 0)
    bits = from_dev(gpu.logits())[0]
    say("  [gpu] sample_token: greedy and top-p on the model's logits")
    assert gpu.sample_token(Sampler(temperature=0.0)) == gpu.sample_greedy()
    decided = 0
    for seed in range(12):
        rand = Sampler(seed=seed).next_rand()
        tok = gpu.sample_token(Sampler(seed=seed, temperature=0.7, top_p=0.9, top_k=50))
        want = orc.sort_and_sample(bits, 0.9, 64, rand)
        assert tok in set(want["keys"].tolist())
        if pins.top_p_closed_form(want["vals"], 0.9, rand)[1] > 1e-5:
            decided += 1
            assert tok == want["token"]
    assert decided >= 6


def test_decode_graph_replays_the_eager_loop(qwen):
    """Qwen2Model.capture_decode: the greedy loop replayed from one HIP graph
    (token and position on the device, no host work per token) gives the eager
    loop's tokens step by step: a 32-token prompt, then 48 greedy steps.  The
    host reads each replay's token before the next replay."""
    cfg, gpu, _ = qwen
    rng = np.random.default_rng(41)
    prompt = rng.integers(0, cfg.vocab_size, 32).tolist()
    gpu.forward(prompt, 0)
    eager = [gpu.sample_greedy()]
    pos = len(prompt)
    for _ in range(48):
        gpu.forward([eager[-1]], pos)
        eager.append(gpu.sample_greedy())
        pos += 1
    gpu.forward(prompt, 0)  # the prompt's cache rows again; the graph rewrites the rest
    assert gpu.sample_greedy() == eager[0]
    say("  [gpu] decode graph: capture, then 48 replays against the eager loop")
    graph = gpu.capture_decode(max_ctx=256)
    gpu.pos.fill_(len(prompt))  # gpu.idx holds the first token
    for s in range(48):
        graph.replay()
        tok = int(gpu.idx.cpu().item())
        assert tok == eager[s + 1], f"replay {s}: token {tok}, eager loop {eager[s + 1]}"
    assert int(gpu.pos.cpu().item()) == len(prompt) + 48
    say(f"  48 replays equal the eager loop's tokens (first {eager[1:6]})")


@pytest.mark.parametrize("rows,hidden,inter", [
    (2, 64, 64), (63, 128, 192), (64, 896, 4864), (65, 192, 512), (700, 896, 4864), (33, 2048, 320),
    (130, 8192, 64), (256, 320, 192), (257, 320, 192), (1023, 192, 512), (1025, 192, 512),
    (1100, 896, 1024)])
def test_prompt_layer_products(luc, rows, hidden, inter):
    """luc_prompt_gemm and luc_prompt_mlp at the edges of their tiles (64 rows,
    64 columns), of the K splits and of the row length, against the same steps in
    f64 with the roundings the kernels state (h, x, gate, up and act in bf16).
    Every product's f32 sum rounds once, so an element may sit one bf16 unit off
    where its exact value lies next to a rounding boundary, and each rounding
    step passes such units on to what follows: 2^-7 of the row's scale bounds
    the largest difference, and 1 / 64 of the elements may differ by more than a unit."""
    gen = torch.Generator(device="cuda").manual_seed(rows + hidden + inter)

    def mk(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=gen, device="cuda") * std + mean).to(torch.bfloat16)

    h, att = mk(rows, hidden), mk(rows, hidden)
    o_w, gu_w = mk(hidden, hidden, std=hidden ** -0.5), mk(2 * inter, hidden, std=hidden ** -0.5)
    down_w = mk(hidden, inter, std=inter ** -0.5)
    n1, n2 = mk(hidden, std=0.1, mean=1.0), mk(hidden, std=0.1, mean=1.0)
    eps = 1e-6
    r = lambda t: t.to(torch.float32).to(torch.bfloat16).double()  # noqa: E731
    norm = lambda t, w: r(t / torch.sqrt((t * t).mean(-1, keepdim=True) + eps) * w.double())  # noqa: E731
    h1 = r(h.double() + att.double() @ o_w.double().t())
    gu = r(norm(h1, n1) @ gu_w.double().t())
    act = r(torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:])
    h2 = r(h1 + act @ down_w.double().t())
    want_x = norm(h2, n2)
    x = torch.empty_like(h)
    ws = torch.full((luc.lib.luc_prompt_mlp_workspace_size(rows, hidden, inter),), 255,
                    dtype=torch.uint8, device="cuda")
    say(f"  [gpu] prompt_mlp rows={rows} hidden={hidden} inter={inter}")
    luc.prompt_mlp(h, att, o_w, n1, eps, gu_w, down_w, n2, x, ws)
    n = (hidden // 2) // 4 * 4 + 4
    y = torch.empty(rows, n, dtype=torch.bfloat16, device="cuda")
    w = mk(n, hidden, std=hidden ** -0.5)
    luc.prompt_gemm(y, att, w)
    torch.cuda.synchronize()
    for name, got, want in (("y", y, r(att.double() @ w.double().t())), ("h", h, h2), ("x", x, want_x)):
        d = (got.double() - want).abs()
        unit = torch.exp2(torch.floor(torch.log2(want.abs().clamp_min(1e-9))) - 7)
        over = float((d > unit).double().mean())
        say(f"  {name}: max {float(d.max()):.3e}, beyond a unit {over:.4f}")
        assert float((d / want.abs().amax(-1, keepdim=True)).max()) <= 2 ** -7, name
        assert over <= 1 / 64, name


@pytest.mark.parametrize("inter", [320, 8320])
def test_prompt_products_agree_with_library_gemms(luc, monkeypatch, inter):
    """A prompt through luc_prompt_gemm / luc_prompt_mlp and through the library
    GEMMs on the same weights: both sum in f32 and round to bf16 at the same
    places, so they differ by the units that another sum order moves.  A row's
    relative error from one such rounding is at most 2^-9 in the 2-norm; a layer
    has seven (norm, q/k/v, attention, h, norm, gate and up, act) before the
    last h, two layers fourteen, and independent ones add as squares: sqrt(14) 2^-9
    = 0.0073, doubled for two paths that round apart."""
    cfg = Qwen2Config(vocab_size=512, hidden_size=256, num_hidden_layers=2, num_attention_heads=4,
                      num_key_value_heads=2, intermediate_size=inter, max_position_embeddings=512)
    w = random_weights(cfg, 5, std=0.06)
    ids = [int(i) for i in np.random.default_rng(6).integers(0, 512, 130)]
    got = []
    for own in (True, False):
        monkeypatch.setattr(model_module, "prompt_kernels_win", lambda cfg, rows, own=own: own)
        m = Qwen2Model(cfg, w, max_positions=256, lib=luc)
        m.forward(ids, 0)
        got.append([t.float() for t in (m.hidden, m.logits(), m.kv.k_pool, m.kv.v_pool)])
    torch.cuda.synchronize()
    for a, b in zip(*got):
        err = float((a - b).norm() / b.norm())
        say(f"  own products against library GEMMs: {err:.2e}")
        assert err <= 2 * 14 ** 0.5 * 2 ** -9
