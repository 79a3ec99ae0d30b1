"""HIP causal prefill (RoPE + cache write + MFMA attention of packed prompts)
vs the oracle, through the C ABI.  Roped q/k (in place) and the cache are
compared bit for bit; attention outputs within the stated tolerance
(max-abs 2e-3 fp16, 1e-2 bf16)."""
import contextlib

import numpy as np
import pytest
import torch

from lucciola_rs_amd import workloads as wl
from lucciola_rs_amd.engine import sm_scale
from gpu_util import TOL, from_dev, max_abs, rope_cache, say, to_dev, ulp_gate

pytestmark = pytest.mark.gpu


def biases(cfg, seed):
    rng = np.random.default_rng(seed)
    d = cfg.head_dim
    return (wl.to_bits(wl.normal(rng, (cfg.hq * d,), 0.5), cfg.dtype),
            wl.to_bits(wl.normal(rng, (cfg.hkv * d,), 0.5), cfg.dtype),
            wl.to_bits(wl.normal(rng, (cfg.hkv * d,), 0.5), cfg.dtype))


def gpu_prefill(luc, h: wl.HostPrefill, layer=0, max_ctx=None, bias=None, scale=None, stream=None,
                num_blocks=None):
    cfg = h.cfg
    d = cfg.head_dim
    rope = rope_cache(luc, d)
    qkv = to_dev(h.qkv, cfg.dtype)
    kp, vp = to_dev(h.k_pool, cfg.dtype), to_dev(h.v_pool, cfg.dtype)
    tables = torch.from_numpy(h.tables).cuda()
    cu = torch.from_numpy(h.cu_seqlens).cuda()
    sp = torch.from_numpy(h.start_pos).cuda()
    total = int(h.cu_seqlens[-1])
    out = torch.full((total, cfg.hq * d), 7.0, dtype=cfg.torch_dtype, device="cuda")
    qb, kb, vb = (None, None, None) if bias is None else (to_dev(x, cfg.dtype) for x in bias)
    max_ctx = h.max_ctx if max_ctx is None else max_ctx
    say(f"  [gpu] paged_prefill {cfg.name} rows={np.diff(h.cu_seqlens).tolist()[:8]} "
        f"starts={h.start_pos.tolist()[:8]} hq={cfg.hq} hkv={cfg.hkv} d={d} {cfg.dtype} "
        f"max_ctx={max_ctx} layer={layer} bias={bias is not None}")
    if stream is not None:
        stream.wait_stream(torch.cuda.current_stream())
    luc.paged_prefill(qkv, qb, kb, vb, rope.cos, rope.sin, kp, vp, tables, cu, sp, total, max_ctx,
                      layer, h.num_layers, cfg.hq, cfg.hkv, d, sm_scale(d) if scale is None else scale,
                      out, stream=stream, num_blocks=num_blocks)
    torch.cuda.synchronize()
    return dict(out=from_dev(out).reshape(total, cfg.hq, d), qkv=from_dev(qkv),
                k_pool=from_dev(kp), v_pool=from_dev(vp))


def oracle_prefill(orc, luc, h: wl.HostPrefill, layer=0, bias=None, scale=None):
    cfg = h.cfg
    rope = rope_cache(luc, cfg.head_dim)
    cos, sin = rope.cos.cpu().numpy(), rope.sin.cpu().numpy()
    qkv, kp, vp = h.qkv.copy(), h.k_pool.copy(), h.v_pool.copy()
    qb, kb, vb = (None, None, None) if bias is None else bias
    out = orc.prefill(qkv, qb, kb, vb, cos, sin, kp, vp, h.tables, h.cu_seqlens, h.start_pos,
                      layer, cfg.hq, cfg.hkv, cfg.head_dim,
                      sm_scale(cfg.head_dim) if scale is None else scale, 16, h.num_layers, cfg.dtype)
    return dict(out=out, qkv=qkv, k_pool=kp, v_pool=vp)


def assert_prefill_matches(orc, got, want, dtype, max_frac=0.5):
    """Bit-exact roped q/k and cache; attention outputs within the stated
    max-abs tolerance and within 4 storage units of the oracle's at the row's
    scale (ulp_gate: measured at most ~2.5), with at most `max_frac` of the
    elements differing at all (measured 18-43%)."""
    assert np.array_equal(got["qkv"], want["qkv"]), "RoPE'd q/k differ"
    assert np.array_equal(got["k_pool"], want["k_pool"]), "K pool differs"
    assert np.array_equal(got["v_pool"], want["v_pool"]), "V pool differs"
    o = orc.to_f32(got["out"], dtype)
    assert np.all(np.isfinite(o)), "non-finite attention output"
    err = max_abs(orc, got["out"], want["out"], dtype)
    say(f"  max|hip - oracle| = {err:.3e} (tol {TOL[dtype]})")
    assert err <= TOL[dtype]
    ulp_gate(orc, got["out"], want["out"], dtype, max_ulps=4, max_frac=max_frac)


SHAPES = [(14, 2, 64), (12, 2, 128), (28, 4, 128)]


@pytest.mark.parametrize("hq,hkv,d", SHAPES, ids=[f"{a}q{b}kv-d{c}" for a, b, c in SHAPES])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_prefill_ragged_prompts_and_prefixes(orc, luc, hq, hkv, d, dtype):
    """Prompts of 37, 64 and 1 rows after cached prefixes of 0, 5 and 130
    tokens (partial pages, a tile boundary, a one-row prompt)."""
    cfg = wl.PrefillConfig("ragged", 3, 0, hq, hkv, d, dtype, 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=7, rows=[37, 64, 1], starts=[0, 5, 130])
    assert_prefill_matches(orc, gpu_prefill(luc, h), oracle_prefill(orc, luc, h), dtype)


@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 6, 7, 8])
def test_prefill_every_group_size(orc, luc, group):
    cfg = wl.PrefillConfig(f"g{group}", 2, 0, 2 * group, 2, 64, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=group, rows=[70, 33], starts=[17, 64])
    assert_prefill_matches(orc, gpu_prefill(luc, h), oracle_prefill(orc, luc, h), "bf16")


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
def test_prefill_with_biases_and_layer(orc, luc, dtype):
    """q/k/v biases (Qwen2 has them) and a non-zero layer of a 3-layer cache."""
    cfg = wl.PrefillConfig("bias", 2, 0, 14, 2, 64, dtype, 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=11, num_layers=3, rows=[100, 29], starts=[3, 200])
    bias = biases(cfg, 12)
    for layer in (0, 2):
        assert_prefill_matches(orc, gpu_prefill(luc, h, layer=layer, bias=bias),
                               oracle_prefill(orc, luc, h, layer=layer, bias=bias), dtype)


@pytest.mark.parametrize("batch", [16, 17, 24])
def test_prefill_many_prompts(orc, luc, batch):
    """Many short ragged prompts, empty ones among them (the first, one in the
    middle and the last): the append kernel's workgroups straddle several
    sequences and its cu_seqlens search skips empty ones."""
    rng = np.random.default_rng(batch)
    rows = rng.integers(1, 40, batch)
    rows[[0, batch // 2, batch - 1]] = 0
    starts = rng.integers(0, 50, batch)
    cfg = wl.PrefillConfig(f"many{batch}", batch, 0, 14, 2, 64, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=batch, rows=rows, starts=starts)
    assert_prefill_matches(orc, gpu_prefill(luc, h), oracle_prefill(orc, luc, h), "bf16")


def test_prefill_4x2048_full(orc, luc):
    """The full prefill shape: 4 prompts x 2048 rows from an empty cache,
    14q/2kv, d=64, bf16, 128 pages per sequence."""
    cfg = wl.PREFILL_CONFIGS["prefill_4x2048"]
    h = wl.host_prefill_inputs(cfg, seed=2048)
    assert_prefill_matches(orc, gpu_prefill(luc, h), oracle_prefill(orc, luc, h), "bf16")


def test_prefill_matches_decode_steps(orc, luc):
    """Prefill of a prompt equals decoding its rows one at a time (the
    reference's own loop): the last row's output and the cache agree with the
    decode path's, within f32 rounding of the two accumulation orders."""
    from lucciola_rs_amd.engine import decode_step
    cfg = wl.PrefillConfig("vs_decode", 1, 0, 14, 2, 64, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=3, rows=[96], starts=[40], poison=False)
    got = gpu_prefill(luc, h)
    rope = rope_cache(luc, 64)
    kp, vp = to_dev(h.k_pool, "bf16"), to_dev(h.v_pool, "bf16")
    tables = torch.from_numpy(h.tables).cuda()
    row = cfg.row
    outs = []
    for i in range(96):
        qkv = to_dev(h.qkv[i: i + 1], "bf16")
        pos = torch.tensor([40 + i], dtype=torch.int32, device="cuda")
        out = torch.empty((1, 14 * 64), dtype=torch.bfloat16, device="cuda")
        ws = luc.workspace(1, 14, 2, 64, 40 + i + 1)
        decode_step(qkv, None, None, None, rope, kp, vp, tables, pos, 40 + i + 1, 0, 1, 14, 2, 64,
                    out, ws, 0, lib=luc)
        outs.append(out)
    torch.cuda.synchronize()
    assert np.array_equal(from_dev(kp), got["k_pool"]) and np.array_equal(from_dev(vp), got["v_pool"])
    dec = np.stack([orc.to_f32(from_dev(o).reshape(14, 64), "bf16") for o in outs])
    pre = orc.to_f32(got["out"], "bf16")
    err = float(np.max(np.abs(dec - pre)))
    say(f"  max|prefill - decode loop| = {err:.3e}")
    assert err <= TOL["bf16"]


def test_prefill_beyond_max_ctx_gives_nan(orc, luc):
    """A sequence whose prompt runs past the host bound max_ctx is flagged
    with NaN outputs; the others are computed normally.  RoPE and the cache
    write still cover every row the table can hold, flagged or not."""
    cfg = wl.PrefillConfig("over", 2, 0, 14, 2, 64, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=5, rows=[50, 20], starts=[0, 100])
    got = gpu_prefill(luc, h, max_ctx=60)  # sequence 1 reaches position 119
    o = orc.to_f32(got["out"], "bf16")
    assert np.all(np.isfinite(o[:50])) and np.all(np.isnan(o[50:]))
    want = oracle_prefill(orc, luc, h)
    assert np.array_equal(got["qkv"], want["qkv"]), "RoPE'd q/k differ"
    assert np.array_equal(got["k_pool"], want["k_pool"]) and np.array_equal(got["v_pool"], want["v_pool"])


def test_prefill_long_prompt_beyond_max_ctx_all_flagged(orc, luc):
    """A flagged prompt longer than the grid's tiles (130 rows against a bound
    of 40) has every one of its rows flagged; the other sequence matches the
    oracle."""
    cfg = wl.PrefillConfig("over_long", 2, 0, 14, 2, 64, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=6, rows=[30, 130], starts=[4, 0])
    got = gpu_prefill(luc, h, max_ctx=40)
    o = orc.to_f32(got["out"], "bf16")
    assert np.all(np.isnan(o[30:]))
    want = oracle_prefill(orc, luc, h)
    assert np.array_equal(got["qkv"], want["qkv"]), "RoPE'd q/k differ"
    assert np.array_equal(got["k_pool"], want["k_pool"]) and np.array_equal(got["v_pool"], want["v_pool"])
    err = float(np.max(np.abs(o[:30] - orc.to_f32(want["out"], "bf16")[:30])))
    assert err <= TOL["bf16"]


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (8, 8, 128), (16, 2, 128)])
@pytest.mark.parametrize("rows,starts", [([1, 36, 37], [895, 128, 0]), ([2, 300], [767, 90]),
                                         ([70], [1978])])
def test_prefill_split_contexts(orc, luc, hq, hkv, d, rows, starts):
    """Contexts cut into K splits: rows that end on, before and past a split
    boundary, a sequence shorter than one split beside longer ones, and a tile
    whose rows lie on both sides of a boundary; the unsplit entry point on the
    same inputs agrees to f32 rounding of the sums plus one storage rounding."""
    cfg = wl.PrefillConfig("split", len(rows), 0, hq, hkv, d, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=sum(rows) + d, rows=rows, starts=starts)
    total = int(h.cu_seqlens[-1])
    need = luc.lib.luc_paged_prefill_workspace_size(len(rows), total, h.max_ctx, hq, hkv, d)
    assert need > 0, "these sizes are meant to split"
    got = gpu_prefill(luc, h)
    assert_prefill_matches(orc, got, oracle_prefill(orc, luc, h), "bf16")
    luc_size = luc.lib.luc_paged_prefill_workspace_size
    try:
        luc.lib.luc_paged_prefill_workspace_size = lambda *a: 0
        split = luc.lib.luc_paged_prefill_split
        luc.lib.luc_paged_prefill_split = lambda *a: luc.lib.luc_paged_prefill(*a[:-2])
        whole = gpu_prefill(luc, h)
    finally:
        luc.lib.luc_paged_prefill_workspace_size, luc.lib.luc_paged_prefill_split = luc_size, split
    for name in ("qkv", "k_pool", "v_pool"):
        assert np.array_equal(got[name], whole[name])
    a, b = orc.to_f32(got["out"], "bf16"), orc.to_f32(whole["out"], "bf16")
    # p and the output round to bf16 (2^-9 each) around different maxima
    assert np.max(np.abs(a - b)) <= 2 ** -7 * np.max(np.abs(b))


@pytest.mark.parametrize("hq,hkv,d,batch,hi", [
    (14, 2, 64, 20, 60), (8, 8, 128, 70, 40), (28, 4, 128, 65, 70), (64, 8, 64, 130, 40),
    (12, 4, 64, 257, 30), (4, 4, 128, 600, 12)])
def test_prefill_loose_bound_same_bits(orc, luc, hq, hkv, d, batch, hi):
    """Ragged prompts (empty ones among them: the first, the last, two in a
    row) under a bound max_ctx that is exact and one that is a hundred times too
    large: the workgroups are dealt differently (all the chunks the bound
    allows; slots dealt by cu_seqlens, at one and at several reads of 64 lengths;
    blocks of 64 (sequence, kv head) pairs with a partial last one) and every
    result is the same, bit for bit.  One sequence past the loose bound is
    flagged, also where it alone has more rows than the others together."""
    rng = np.random.default_rng(batch)
    rows = rng.integers(1, hi, batch)
    rows[[0, batch // 2, batch // 2 + 1, batch - 1]] = 0
    cfg = wl.PrefillConfig("loose", batch, 0, hq, hkv, d, "bf16", 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=batch, rows=rows, starts=rng.integers(0, 20, batch))
    tight = gpu_prefill(luc, h)
    wide = wl.replace(h, tables=np.pad(h.tables, ((0, 0), (0, 100 * hi // 16)),
                                       constant_values=int(h.tables.max())))
    loose = gpu_prefill(luc, wide, max_ctx=100 * hi)
    for name in tight:
        assert np.array_equal(tight[name], loose[name]), name
    o = orc.to_f32(tight["out"], "bf16")
    assert np.all(np.isfinite(o))
    # the last sequence now longer than the bound
    rows[-1] = 100 * hi + 7
    h = wl.host_prefill_inputs(cfg, seed=batch, rows=rows, starts=np.zeros(batch, int), poison=False)
    got = gpu_prefill(luc, h, max_ctx=100 * hi)
    o = orc.to_f32(got["out"], "bf16")
    n = int(h.cu_seqlens[-2])
    assert np.all(np.isfinite(o[:n])) and np.all(np.isnan(o[n:]))


def test_prefill_many_prompts_under_a_long_bound(orc, luc):
    """1024 prompts of 32 rows, 64 and 8 heads, and a bound of all the rows in
    one sequence: more than 2^32 threads, were every sequence given the chunks
    that the bound allows.  The same bits as under the exact bound."""
    cfg = wl.PrefillConfig("bound", 1024, 32, 64, 8, 64, "bf16", 0, 0, 0.5)
    gen = torch.Generator(device="cuda").manual_seed(4)
    qkv = torch.randn(1024 * 32, cfg.row, generator=gen, device="cuda").to(torch.bfloat16)
    tables = torch.zeros(1024, 32768 // 16, dtype=torch.int32, device="cuda")
    tables[:, :2] = torch.randperm(2048, generator=gen, device="cuda").to(torch.int32).view(1024, 2)
    cu = torch.arange(1025, dtype=torch.int32, device="cuda") * 32
    start = torch.zeros(1024, dtype=torch.int32, device="cuda")
    rope = rope_cache(luc, 64)
    results = []
    for max_ctx in (32, 32768):
        x, out = qkv.clone(), torch.zeros(1024 * 32, 64 * 64, dtype=torch.bfloat16, device="cuda")
        pools = [torch.zeros(2048, 1, 8, 16, 64, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        say(f"  [gpu] paged_prefill 1024 x 32 rows, max_ctx={max_ctx}")
        luc.paged_prefill(x, None, None, None, rope.cos, rope.sin, *pools, tables, cu, start,
                          1024 * 32, max_ctx, 0, 1, 64, 8, 64, sm_scale(64), out)
        torch.cuda.synchronize()
        results.append([x, out, *pools])
    assert torch.isfinite(results[0][1]).all() and results[0][1].any(-1).all()
    for a, b in zip(*results):
        assert torch.equal(a, b)


@contextlib.contextmanager
def unsplit(luc):
    """luc_paged_prefill, which cuts no contexts, in the place of luc_paged_prefill_split."""
    size, split = luc.lib.luc_paged_prefill_workspace_size, luc.lib.luc_paged_prefill_split
    try:
        luc.lib.luc_paged_prefill_workspace_size = lambda *a: 0
        luc.lib.luc_paged_prefill_split = lambda *a: luc.lib.luc_paged_prefill(*a[:-2])
        yield
    finally:
        luc.lib.luc_paged_prefill_workspace_size, luc.lib.luc_paged_prefill_split = size, split


@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("hq,hkv,d", [(4, 4, 64), (14, 2, 64), (8, 8, 128), (12, 2, 128), (32, 4, 128)])
def test_prefill_unsplit_at_chunk_edges(orc, luc, hq, hkv, d, dtype):
    """Whole contexts, as luc_paged_prefill takes them, on 4-wave workgroups (so few
    rows leave CUs idle): prompts that end one column of a 128-column chunk
    before its end, on it and past it (where the group size divides it), after
    prefixes that end on and around a 64-token block, with biases, in layer 2 of 3."""
    g = hq // hkv
    cfg = wl.PrefillConfig("edges", 4, 0, hq, hkv, d, dtype, 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=hq + d, num_layers=3, starts=[0, 63, 64, 130],
                               rows=[128 // g, 256 // g + 1, 128 // g - 1, 3])
    bias = biases(cfg, 13)
    with unsplit(luc):
        got = gpu_prefill(luc, h, layer=2, bias=bias)
    assert_prefill_matches(orc, got, oracle_prefill(orc, luc, h, layer=2, bias=bias), dtype)


def split_prefill(hq, hkv, d, dtype, rows, starts, seed, luc, max_ctx=None, **kw):
    """Inputs whose contexts the plan cuts."""
    cfg = wl.PrefillConfig("split", len(rows), 0, hq, hkv, d, dtype, 0, 0, 0.5)
    h = wl.host_prefill_inputs(cfg, seed=seed, rows=rows, starts=starts, **kw)
    need = luc.lib.luc_paged_prefill_workspace_size(len(rows), int(h.cu_seqlens[-1]),
                                                    max_ctx or h.max_ctx, hq, hkv, d)
    assert need > 0, "these sizes are meant to split"
    return h


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (12, 2, 128)])
@pytest.mark.parametrize("dtype", ["bf16", "f16"])
@pytest.mark.parametrize("sign", [1.0, -1.0])
def test_prefill_split_with_biases_and_layer(orc, luc, hq, hkv, d, dtype, sign):
    """Cut contexts with q, k and v biases, in layers 0 and 2 of 3, in both dtypes and
    with a negative score scale, on a stream of its own (whose workspace the wrapper
    allocates there) while the current one is another."""
    h = split_prefill(hq, hkv, d, dtype, [300, 1, 90], [600, 880, 0], 31, luc, num_layers=3)
    bias = biases(h.cfg, 32)
    stream = torch.cuda.Stream()
    for layer in (0, 2):
        want = oracle_prefill(orc, luc, h, layer=layer, bias=bias, scale=sign * sm_scale(d))
        assert_prefill_matches(orc, gpu_prefill(luc, h, layer=layer, bias=bias, scale=sign * sm_scale(d)),
                               want, dtype)
        got = gpu_prefill(luc, h, layer=layer, bias=bias, scale=sign * sm_scale(d), stream=stream)
        assert_prefill_matches(orc, got, want, dtype)


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (12, 2, 128)])
def test_prefill_split_page_outside_the_pool(orc, luc, hq, hkv, d):
    """A table entry outside the pool that only one split of several sees (tokens
    640..655 of 900): the rows before it match the oracle, the rows at and after it
    are NaN, in that split and in the next, and the other sequence is untouched."""
    h = split_prefill(hq, hkv, d, "bf16", [300, 90], [600, 700], 33, luc, poison=False)
    want = oracle_prefill(orc, luc, h)
    tables = h.tables.copy()
    tables[0, 40] = h.k_pool.shape[0] + 1
    spare = np.zeros((4,) + h.k_pool.shape[1:], np.uint16)
    bad = wl.replace(h, tables=tables, k_pool=np.concatenate([h.k_pool, spare]),
                     v_pool=np.concatenate([h.v_pool, spare]))
    got = gpu_prefill(luc, bad, num_blocks=h.k_pool.shape[0])
    o, w = orc.to_f32(got["out"], "bf16"), orc.to_f32(want["out"], "bf16")
    ok = np.r_[np.arange(300) < 40, np.ones(90, bool)]
    assert np.all(np.isnan(o[~ok]))
    assert np.max(np.abs(o[ok] - w[ok])) <= TOL["bf16"]
    assert not got["k_pool"][-4:].any() and not got["v_pool"][-4:].any()
    assert np.array_equal(got["qkv"], want["qkv"])


@pytest.mark.parametrize("hq,hkv,d", [(14, 2, 64), (12, 2, 128)])
def test_prefill_split_beside_a_flagged_sequence(orc, luc, hq, hkv, d):
    """A sequence past max_ctx between two whose contexts are cut: NaN in all of its
    rows (and no later split or merge writes there), the oracle's results in theirs."""
    h = split_prefill(hq, hkv, d, "bf16", [200, 50, 100], [600, 1200, 650], 34, luc, max_ctx=800)
    got = gpu_prefill(luc, h, max_ctx=800)
    want = oracle_prefill(orc, luc, h)
    o, w = orc.to_f32(got["out"], "bf16"), orc.to_f32(want["out"], "bf16")
    assert np.all(np.isnan(o[200:250]))
    for rows in (slice(0, 200), slice(250, 350)):
        assert np.max(np.abs(o[rows] - w[rows])) <= TOL["bf16"]
    for name in ("qkv", "k_pool", "v_pool"):
        assert np.array_equal(got[name], want[name]), name
