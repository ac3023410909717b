"""Batched prefill on the MI355X: the Q4_0 MFMA GEMM against the oracle's
per-row GEMV, and the batched prompt phase against the oracle's per-token
forward loop (the reference's own prompt phase, src/model/mod.rs:57-125).

Bars:
  * GEMM: max|y - y_oracle| / max|y_oracle| <= 1e-4 (f32 accumulate) and, per
    element, |y - y_f64| <= 2e-5 * sum_k |w_k x_k|.
  * Prefill: logits of the last prompt position within 1e-3 absolute of the
    oracle's, the same next token, and greedy ids identical when decoding
    continues from the prefilled cache.
"""
import numpy as np
import pytest

import cw
import oracle as orc

pytestmark = pytest.mark.gpu

LOGIT_TOL = 1e-3


def rel_err(y, ref):
    return float(np.max(np.abs(y.astype(np.float64) - ref)) / max(np.max(np.abs(ref)), 1e-30))


GEMM_SHAPES = [  # (m, in_f, out_f)
    (1, 256, 512), (7, 1024, 3072), (64, 4096, 256), (65, 2048, 1024), (37, 96, 100),
    (130, 160, 65), (512, 4096, 512), (200, 12288, 128), (3, 32, 7),
    (100, 4160, 200),  # K split in two halves of 65 blocks (odd: a half-empty last stage)
]


@pytest.mark.parametrize("m,in_f,out_f", GEMM_SHAPES)
def test_q4_gemm_vs_oracle(ctx, m, in_f, out_f):
    s, q = cw.synth_q4(cw.synth_key(21, f"g{out_f}x{in_f}"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(21, f"gx{m}x{in_f}"), m * in_f).reshape(m, in_f)
    y = ctx.q4_gemm(ctx.storage(x), m, ctx.storage(s), ctx.storage(q), in_f, out_f).download()
    y = y.reshape(m, out_f)
    orc.set_threads(8)
    worst = 0.0
    for i in range(m):
        ref = orc.q4_gemv(x[i], s, q, in_f, out_f)
        worst = max(worst, rel_err(y[i], ref))
        y64, absy = orc.q4_gemv_f64(x[i], s, q, in_f, out_f)
        assert np.all(np.abs(y[i] - y64) <= 2e-5 * absy + 1e-30), i
    assert worst <= 1e-4, worst


# Edges of the GEMM's tiles (16, 32 and 64 rows; 64, 128 and 256 columns), of
# its scale groups (8 blocks) and K splits, one row and one column included
GEMM_EDGES = [(m, k, n) for m in (1, 15, 17, 33, 63, 65, 129)
              for k, n in ((32, 1), (288, 63), (2048, 129))] + \
             [(2, 12288, 65), (16, 40960, 64), (31, 4128, 257), (260, 1024, 300),
              (513, 12288, 4096)]


@pytest.mark.parametrize("m,in_f,out_f", GEMM_EDGES)
def test_q4_gemm_tile_edges(ctx, m, in_f, out_f):
    """Every element against an f64 product of the exactly dequantized
    weights.  The operands are exact to 2^-23 and the sums are f32: the same
    bound as above, 2e-5 * sum_k |w x| (at most 15 + 80 + 15 additions of 2^-24
    in a chain of 16 blocks, the chains of 1,280 blocks and 16 K splits, and two
    more in a block's sum: 6.7e-6)."""
    s, q = cw.synth_q4(cw.synth_key(25, f"e{out_f}x{in_f}"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(25, f"ex{m}x{in_f}"), m * in_f).reshape(m, in_f)
    y = ctx.q4_gemm(ctx.storage(x), m, ctx.storage(s), ctx.storage(q), in_f, out_f).download()
    w = orc.dequant_q4_0_soa(s, q).reshape(out_f, in_f).astype(np.float64)
    x64 = x.astype(np.float64)
    err = np.abs(y.reshape(m, out_f) - x64 @ w.T)
    assert np.all(err <= 2e-5 * (np.abs(x64) @ np.abs(w).T) + 1e-30)


@pytest.mark.parametrize("m,in_f,out_f", [(4, 288, 512), (1, 32, 33000), (1000, 288, 513),
                                          (3, 1056, 40000), (1030, 2080, 300)])
def test_q4_gemm_padded_scales_take_no_launch(ctx, m, in_f, out_f):
    """Scale rows that are not whole groups of eight blocks are copied by the
    pass that splits x, by its own workgroups, few or many beside the rows':
    no launch more than aligned rows take, and results within
    2e-5 * sum_k |w x| of 64 bits."""
    s, q = cw.synth_q4(cw.synth_key(29, f"p{out_f}x{in_f}"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(29, f"px{m}x{in_f}"), m * in_f).reshape(m, in_f)
    dev = [ctx.storage(v) for v in (x, s, q)]
    ctx.profile_begin()
    y = ctx.q4_gemm(dev[0], m, dev[1], dev[2], in_f, out_f).download().reshape(m, out_f)
    launches = {r[0]: r[1] for r in ctx.profile_report()}
    assert launches in ({"prefill_split": 1, "q4_gemm": 1},
                        {"prefill_split": 1, "q4_gemm_splitk": 1, "q4_gemm_reduce": 1}), launches
    rows = np.unique(np.linspace(0, m - 1, 30).astype(int))
    w = orc.dequant_q4_0_soa(s, q).reshape(out_f, in_f).astype(np.float64)
    x64 = x[rows].astype(np.float64)
    err = np.abs(y[rows] - x64 @ w.T)
    assert np.all(err <= 2e-5 * (np.abs(x64) @ np.abs(w).T) + 1e-30)


# Rows of x in long segments, whose split keeps six chunks a thread (segments of
# over 4,096 elements, four rows a workgroup) or reads the rest of a segment
# above 12,288 elements again (by one row and by four); with the launches that
# show how the plan splits K (not at all: the segment is the whole row)
GEMM_LONG_ROWS = [(64, 65568, 70, "q4_gemm_splitk"), (1030, 12320, 70, "q4_gemm_splitk"),
                  (900, 12800, 6144, "q4_gemm"), (1500, 12800, 4096, "q4_gemm")]


@pytest.mark.parametrize("m,in_f,out_f,launch", GEMM_LONG_ROWS)
def test_q4_gemm_long_rows(ctx, m, in_f, out_f, launch):
    """Sampled rows and columns (the last of each among them) within
    2e-5 * sum_k |w x| of 64 bits, as above."""
    rng = np.random.default_rng(28)
    s = np.abs(0.02 * rng.standard_normal((out_f, in_f // 32), np.float32)).astype(np.float16)
    q = rng.integers(0, 256, (out_f, in_f // 32, 16), np.uint8)
    x = rng.standard_normal((m, in_f), np.float32)
    dev = [ctx.storage(v) for v in (x, s.view(np.uint16), q)]
    ctx.profile_begin()
    y = ctx.q4_gemm(dev[0], m, dev[1], dev[2], in_f, out_f).download().reshape(m, out_f)
    labels = [r[0] for r in ctx.profile_report()]
    for d in dev:
        ctx.free(d)
    assert launch in labels, labels
    rows = np.unique(np.linspace(0, m - 1, 40).astype(int))
    cols = np.unique(np.linspace(0, out_f - 1, 70).astype(int))
    w = orc.dequant_q4_0_soa(s[cols].view(np.uint16), q[cols]).reshape(len(cols), in_f)
    w, x = w.astype(np.float64), x[rows].astype(np.float64)
    err = np.abs(y[np.ix_(rows, cols)] - x @ w.T)
    assert np.all(err <= 2e-5 * (np.abs(x) @ np.abs(w).T))


def test_q4_gemm_scales_at_odd_addresses(ctx):
    """Scales at an address that is a multiple of 2 only give the same bits as
    aligned ones (they are copied to aligned rows first)."""
    m, in_f, out_f = 20, 512, 96
    s, q = cw.synth_q4(cw.synth_key(26, "w"), out_f, in_f, 0.02)
    x = ctx.storage(cw.synth_normal_f32(cw.synth_key(26, "x"), m * in_f))
    qd = ctx.storage(q)
    ref = ctx.q4_gemm(x, m, ctx.storage(s), qd, in_f, out_f).download()
    moved = ctx.storage(np.concatenate([np.zeros(1, np.uint16), s.reshape(-1)]))
    at2 = cw.DeviceArray(ctx, s.shape, np.uint16, moved.ptr + 2)
    assert np.array_equal(ref, ctx.q4_gemm(x, m, at2, qd, in_f, out_f).download())


@pytest.mark.parametrize("m,in_f,out_f", [(2, 4096, 4096), (60, 4096, 4096), (384, 4096, 12288),
                                          (1000, 4096, 6144), (700, 12288, 4096),
                                          (1500, 12288, 4096)])
def test_q4_gemm_error_whatever_the_k_splits(ctx, m, in_f, out_f):
    """The 2-norm error of sampled rows against 64 bits, for plans that split K
    much (few rows) and not at all (many).  With one rounding of 2^-24 at most
    per f32 sum, uniform in size (variance 2^-48 / 3, half of it over a binade)
    and relative to a random walk's partial sum, chains of 16 blocks and the
    sum of the chains have the variance 2^-48 / 6 (16 + blocks / 16) / 2; the
    operands and block sums add (0.8e-7)^2 (measured at one block).  The bound
    is 1.25 times that; one chain over all of K had 1.8 to 2.6 times."""
    s, q = cw.synth_q4(cw.synth_key(27, f"c{out_f}x{in_f}"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(27, f"cx{m}x{in_f}"), m * in_f).reshape(m, in_f)
    y = ctx.q4_gemm(ctx.storage(x), m, ctx.storage(s), ctx.storage(q), in_f, out_f).download()
    rows = np.unique(np.linspace(0, m - 1, 24).astype(int))
    w = orc.dequant_q4_0_soa(s, q).reshape(out_f, in_f).astype(np.float64)
    ref = x[rows].astype(np.float64) @ w.T
    err = np.linalg.norm(y.reshape(m, out_f)[rows] - ref) / np.linalg.norm(ref)
    var = 2.0 ** -48 / 6 * (16 + in_f / 512) / 2 + 0.8e-7 ** 2
    assert err <= 1.25 * var ** 0.5, (err, var ** 0.5)


# the four projection shapes of one 8B layer at the 512-token workload:
# QKV (4096 -> 6144), O (4096 -> 4096), gate/up (4096 -> 12288, each) and
# down (12288 -> 4096); (m, in_f, out_f).  These run the split-K and tile
# choices the prefill bench times.
GEMM_8B_512 = [(512, 4096, 6144), (512, 4096, 4096), (512, 4096, 12288), (512, 12288, 4096)]


@pytest.mark.parametrize("m,in_f,out_f", GEMM_8B_512)
def test_q4_gemm_8b_shapes_at_512(ctx, m, in_f, out_f):
    """Every element against an f64 product of the exactly dequantized
    weights (|y - y64| <= 2e-5 * sum_k |w x|, and 1e-4 of max|y| overall);
    sample rows against the oracle's sequential dot (main.rs:133-150)."""
    s, q = cw.synth_q4(cw.synth_key(23, f"g{out_f}x{in_f}"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(23, f"gx{m}x{in_f}"), m * in_f).reshape(m, in_f)
    y = ctx.q4_gemm(ctx.storage(x), m, ctx.storage(s), ctx.storage(q), in_f, out_f).download()
    y = y.reshape(m, out_f).astype(np.float64)
    w = orc.dequant_q4_0_soa(s, q).reshape(out_f, in_f).astype(np.float64)
    x64 = x.astype(np.float64)
    y64 = x64 @ w.T
    bound = np.abs(x64) @ np.abs(w).T
    err = np.abs(y - y64)
    worst = np.unravel_index(np.argmax(err / (bound + 1e-30)), err.shape)
    assert np.all(err <= 2e-5 * bound + 1e-30), (worst, err[worst], bound[worst])
    rel = float(np.max(err) / np.max(np.abs(y64)))
    print(f"\n[q4_gemm {m}x{in_f}->{out_f}] max rel err vs f64 {rel:.2e}", flush=True)
    assert rel <= 1e-4
    orc.set_threads(16)
    for i in (0, 1, 63, 64, 127, 128, 255, 256, 383, 511):
        ref = orc.q4_gemv(x[i], s, q, in_f, out_f)
        assert rel_err(y[i], ref) <= 1e-4, i


def test_q4_gemm_rows_match_gemv(ctx):
    """Every row of the batched GEMM equals the decode GEMV of that row to
    within the same tolerance (two different kernels, one definition)."""
    m, in_f, out_f = 20, 4096, 1024
    s, q = cw.synth_q4(cw.synth_key(22, "w"), out_f, in_f, 0.02)
    x = cw.synth_normal_f32(cw.synth_key(22, "x"), m * in_f).reshape(m, in_f)
    sd, qd = ctx.storage(s), ctx.storage(q)
    y = ctx.q4_gemm(ctx.storage(x), m, sd, qd, in_f, out_f).download().reshape(m, out_f)
    for i in range(m):
        g = ctx.q4_gemv(ctx.storage(x[i]), sd, qd, in_f, out_f).download()
        assert rel_err(y[i], g.astype(np.float64)) <= 1e-4, i


def test_q4_gemm_large_scales(ctx):
    """Block scales up to the f16 maximum (and the smallest subnormal) go
    through the GEMM as they do through the oracle's GEMV: each block's f32
    sum times d."""
    m, in_f, out_f = 37, 512, 96
    s, q = cw.synth_q4(cw.synth_key(24, "w"), out_f, in_f, 0.02)
    big = np.array([8192.0, -30000.0, 65504.0, -65504.0, 2.0 ** -24], np.float16).view(np.uint16)
    rng = np.random.default_rng(24)
    pick = rng.integers(0, s.size, 200)
    s.reshape(-1)[pick] = big[np.arange(200) % big.size]
    x = cw.synth_normal_f32(cw.synth_key(24, "x"), m * in_f).reshape(m, in_f)
    y = ctx.q4_gemm(ctx.storage(x), m, ctx.storage(s), ctx.storage(q), in_f, out_f).download()
    y = y.reshape(m, out_f)
    assert np.all(np.isfinite(y))
    for i in range(m):
        y64, absy = orc.q4_gemv_f64(x[i], s, q, in_f, out_f)
        assert np.all(np.abs(y[i] - y64) <= 2e-5 * absy + 1e-30), i
        assert rel_err(y[i], orc.q4_gemv(x[i], s, q, in_f, out_f)) <= 1e-4, i


def test_q4_gemm_argument_errors(ctx):
    s, q = cw.synth_q4(cw.synth_key(1, "e"), 64, 64, 0.02)
    x = ctx.storage(np.zeros((2, 64), np.float32))
    sd, qd = ctx.storage(s), ctx.storage(q)
    with pytest.raises(cw.CwError):
        ctx.q4_gemm(x, 2, sd, qd, 48, 64)   # in_f not a multiple of 32
    with pytest.raises(cw.CwError):
        ctx.q4_gemm(x, 0, sd, qd, 64, 64)   # no rows


def test_model_rejects_non_finite_scales(ctx):
    """A projection block scale that is not finite is refused at upload;
    large finite ones (8192, the f16 maximum) are accepted."""
    cfg = cw.make_config(1, 64, 2, 1, 32, 64, 100, 8, cw.CW_F16)
    m = cw.Model(ctx, cfg)
    s, q = cw.synth_q4(cw.synth_key(3, "w"), 64, 64, 0.02)
    for bad in (0x7C00, 0xFC00, 0x7E00, 0xFE01):   # +inf, -inf, NaNs
        s2 = s.copy()
        s2[5, 1] = bad
        with pytest.raises(cw.CwError, match="block 11"):
            m.set_weights({"blk.0.attn_q.weight": (s2, q)})
    for big in (0x7000, 0xF000, 0x7BFF):   # 8192, -8192, 65504
        s2 = s.copy()
        s2[5, 1] = big
        m.set_weights({"blk.0.attn_q.weight": (s2, q)})
    m.set_weights({"blk.0.attn_q.weight": (s, q)})
    m.close()


def small_f16(max_seq, n_layers=2, dim=256, n_heads=4, n_kv=2, hidden=512, vocab=1000):
    return cw.make_config(n_layers, dim, n_heads, n_kv, 128, hidden, vocab, max_seq, cw.CW_F16,
                          1e-6, 1e6)


def oracle_prompt_logits(o, prompt, start=0):
    logits = None
    for i, t in enumerate(prompt):
        logits, _ = o.step(int(t), start + i)
    return logits


@pytest.mark.parametrize("P", [1, 5, 64, 100])
def test_prefill_small_model(ctx, P):
    """Batched prompt phase of P tokens (ragged and whole 64-position tiles)
    against the oracle's per-token forward, then 12 greedy decode steps from
    the prefilled cache against the oracle's generate."""
    N = 12
    cfg = small_f16(P + N + 1)
    weights = cw.synthetic_weights(cfg, 77)
    prompt = cw.synth_tokens(cw.synth_key(77, f"p{P}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    ref_logits = oracle_prompt_logits(o, prompt)
    diff = float(np.max(np.abs(m.logits() - ref_logits)))
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref_logits))
    m.decode_async(N, mode=cw.STEP_GRAPH)
    toks = m.tokens(N)
    ref, margins = o.generate(prompt, N + 1)
    assert int(ref[0]) == nxt
    assert np.array_equal(toks, ref[1:N + 1]), (toks, ref[1:N + 1])
    m.close()
    o.close()


@pytest.mark.parametrize("P", [2, 20, 40, 70])
def test_prefill_odd_widths(ctx, P):
    """Widths that are not whole scale groups (288 and 544: 9 and 17 blocks)
    through every projection, for prompts on either side of the 16, 32 and 64
    row tiles: logits within 1e-3 of the oracle's per-token forward."""
    cfg = small_f16(P + 2, dim=288, hidden=544)
    weights = cw.synthetic_weights(cfg, 82)
    prompt = cw.synth_tokens(cw.synth_key(82, f"p{P}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    ref_logits = oracle_prompt_logits(o, prompt)
    diff = float(np.max(np.abs(m.logits() - ref_logits)))
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref_logits))
    m.close()
    o.close()


def test_prefill_after_a_longer_one(ctx):
    """A shorter prompt through the buffers of a longer one (its plans split K
    further) gives the logits of a fresh model's."""
    cfg = small_f16(300)
    weights = cw.synthetic_weights(cfg, 83)
    prompt = cw.synth_tokens(cw.synth_key(83, "p"), 280, cfg.vocab)
    logits = []
    for first in (280, 0):
        m = cw.Model(ctx, cfg)
        m.set_weights(weights)
        m.finalize()
        if first:
            m.prefill(prompt)
        m.prefill(prompt[:150])
        logits.append(m.logits())
        m.close()
    assert float(np.max(np.abs(logits[0] - logits[1]))) <= 1e-4


@pytest.mark.parametrize("P,launch", [(3, "q4_gemm_reduce_split"), (40, "prefill_split_rmsnorm")])
def test_prefill_rows_above_12288(ctx, P, launch):
    """A hidden state wider than the 12,288 elements that the split passes keep
    in registers: the embedding pass, the sum of partials (few rows) and the
    plain normalised split (more rows) read or store the rest of a row twice.
    Logits within 1e-3 of the oracle's."""
    cfg = cw.make_config(1, 12832, 4, 2, 128, 1024, 300, 48, cw.CW_F32, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 88)
    prompt = cw.synth_tokens(cw.synth_key(88, f"p{P}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    ctx.profile_begin()
    nxt = m.prefill(prompt)
    labels = [r[0] for r in ctx.profile_report()]
    assert launch in labels, labels
    o = orc.OracleModel(cfg, weights)
    ref = oracle_prompt_logits(o, prompt)
    o.close()
    diff = float(np.max(np.abs(m.logits() - ref)))
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref))
    m.close()


@pytest.mark.parametrize("kv,tol", [(cw.CW_F16, LOGIT_TOL), (cw.CW_F32, 2e-5)])
@pytest.mark.parametrize("P", [4097, 4133])
def test_prefill_beyond_one_chunk(ctx, kv, tol, P):
    """A prompt longer than the 4,096 positions of one pass (the rest one row,
    and several): the logits of the same prompt in two calls of fewer (f32 sums
    in another order; with an f16 cache also ties), and generate's first id."""
    cfg = cw.make_config(1, 256, 4, 2, 128, 512, 500, 4200, kv, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 89)
    prompt = cw.synth_tokens(cw.synth_key(89, f"p{P}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    nxt = m.prefill(prompt)
    logits = m.logits()
    assert m.generate(prompt, 2)[0] == nxt
    m.prefill(prompt[:2000])
    assert m.prefill(prompt[2000:], start_pos=2000) == nxt
    diff = float(np.max(np.abs(m.logits() - logits)))
    m.close()
    assert diff <= tol, diff


@pytest.mark.parametrize("n_heads,n_kv", [(4, 4), (8, 1), (16, 2)])
def test_prefill_query_groupings(ctx, n_heads, n_kv):
    """The batched prompt phase (130 positions: two whole 64-position tiles
    and a ragged one) with one and with eight query heads per kv head: last
    position's logits within 1e-3 of the oracle's per-token forward, the same
    next token, then 8 greedy decode steps from the prefilled cache."""
    P, N = 130, 8
    cfg = small_f16(P + N + 1, n_heads=n_heads, n_kv=n_kv)
    weights = cw.synthetic_weights(cfg, 78 + n_heads + n_kv)
    prompt = cw.synth_tokens(cw.synth_key(78, f"q{n_heads}x{n_kv}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    ref_logits = oracle_prompt_logits(o, prompt)
    diff = float(np.max(np.abs(m.logits() - ref_logits)))
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref_logits))
    m.decode_async(N, mode=cw.STEP_GRAPH)
    toks = m.tokens(N)
    ref, _ = o.generate(prompt, N + 1)
    assert int(ref[0]) == nxt
    assert np.array_equal(toks, ref[1:N + 1]), (toks, ref[1:N + 1])
    m.close()
    o.close()


def test_prefill_in_chunks_equals_one_pass(ctx):
    """Two prefill calls (positions 0..39, then 40..99 over the cache the
    first wrote) leave the same logits and next token as one 100-position
    call: attention of a later chunk reads the earlier rows from the cache."""
    cfg = small_f16(128)
    weights = cw.synthetic_weights(cfg, 78)
    prompt = cw.synth_tokens(cw.synth_key(78, "p"), 100, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    a = m.prefill(prompt)
    la = m.logits()
    m.prefill(prompt[:40])
    b = m.prefill(prompt[40:], start_pos=40)
    lb = m.logits()
    assert a == b
    assert float(np.max(np.abs(la - lb))) <= 1e-4
    m.close()


def test_prefill_qwen3_8b_layers(ctx):
    """Two layers of the Qwen3-8B shape (hidden 4096, 32/8 heads x 128,
    intermediate 12288; vocab cut to 4096 so the oracle finishes quickly):
    a 96-token batched prefill against the oracle's per-token loop, then 8
    greedy steps."""
    P, N = 96, 8
    cfg = cw.make_config(2, 4096, 32, 8, 128, 12288, 4096, P + N + 1, cw.CW_F16, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 80)
    prompt = cw.synth_tokens(cw.synth_key(80, "p"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    orc.set_threads(16)
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    ref_logits = oracle_prompt_logits(o, prompt)
    diff = float(np.max(np.abs(m.logits() - ref_logits)))
    print(f"\n[qwen3-8b x2 layers] prefill {P}: max |logit diff| = {diff:.3e}", flush=True)
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref_logits))
    m.decode_async(N, mode=cw.STEP_GRAPH)
    toks = m.tokens(N)
    ref, _ = o.generate(prompt, N + 1)
    assert np.array_equal(toks, ref[1:N + 1]), (toks, ref[1:N + 1])
    m.close()
    o.close()


def test_prefill_qwen3_8b_layers_512(ctx):
    """The benchmarked prompt length: a 512-token batched prefill on two
    layers of the Qwen3-8B shape (vocab cut to 4096 so the oracle's 512
    per-token forwards finish quickly).  Causal MFMA attention over 8 query
    tiles and 512 keys, the M = 512 split-K GEMMs with the in-place residual:
    last-position logits within 1e-3 of the oracle's per-token loop, the same
    next token, then 4 greedy steps from the prefilled cache."""
    P, N = 512, 4
    cfg = cw.make_config(2, 4096, 32, 8, 128, 12288, 4096, P + N + 1, cw.CW_F16, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 81)
    prompt = cw.synth_tokens(cw.synth_key(81, "p512"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    orc.set_threads(16)
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    gl = m.logits()
    ref_logits = oracle_prompt_logits(o, prompt)
    diff = float(np.max(np.abs(gl - ref_logits)))
    top = np.sort(ref_logits)[-2:]
    print(f"\n[qwen3-8b x2 layers] prefill {P}: max |logit diff| = {diff:.3e}, "
          f"oracle top-2 margin {top[1] - top[0]:.3e}", flush=True)
    assert diff <= LOGIT_TOL, diff
    assert nxt == int(np.argmax(ref_logits))
    m.decode_async(N, mode=cw.STEP_GRAPH)
    toks = m.tokens(N)
    # the oracle continues from its own cache (rows 0..P-1 written above)
    ref, t = [], nxt
    for i in range(N):
        lg, _ = o.step(int(t), P + i)
        t = int(np.argmax(lg))
        ref.append(t)
    assert np.array_equal(toks, np.array(ref, np.uint32)), (toks, ref)
    m.close()
    o.close()


@pytest.mark.parametrize("kv", [cw.CW_F16, cw.CW_F32])
@pytest.mark.parametrize("n_heads,n_kv", [(4, 4), (4, 2), (8, 2), (8, 1)])
def test_prefill_attention_chunks(ctx, kv, n_heads, n_kv):
    """The prompt phase behind a filled cache, at the edges of attention's
    query tiles (16 positions a wave) and key tiles (64 keys, 32 for f32) and
    with its keys in many chunks: logits within 1e-3 of the oracle's per-token
    forward over the same cache."""
    cfg = cw.make_config(1, 256, n_heads, n_kv, 128, 512, 500, 460, kv, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 84 + n_heads + n_kv)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    es = np.float16 if kv == cw.CW_F16 else np.float32
    rng = np.random.default_rng(84)
    for start, P in ((0, 2), (0, 33), (0, 129), (31, 16), (63, 17), (64, 65), (333, 3),
                     (389, 70)):
        k, v = (rng.standard_normal((1, max(start, 1), n_kv * 128)).astype(es) for _ in range(2))
        prompt = cw.synth_tokens(cw.synth_key(84, f"a{start}x{P}"), P, cfg.vocab)
        o = orc.OracleModel(cfg, weights)
        if start:
            bits = np.uint16 if kv == cw.CW_F16 else np.float32
            m.prefill_kv(k.view(bits), v.view(bits), start)
            o.prefill_kv(k.view(bits), v.view(bits), start)
        nxt = m.prefill(prompt, start_pos=start)
        ref = oracle_prompt_logits(o, prompt, start)
        diff = float(np.max(np.abs(m.logits() - ref)))
        assert diff <= LOGIT_TOL, (start, P, diff)
        assert nxt == int(np.argmax(ref)), (start, P)
        o.close()
    m.close()


@pytest.mark.parametrize("n_heads,n_kv", [(4, 2), (4, 1)])
@pytest.mark.parametrize("start,P", [(60, 3), (60, 40), (400, 3), (400, 40)])
def test_prefill_attention_behind_a_sink(ctx, n_heads, n_kv, start, P):
    """One key 12 to 16 nats above all others whose V row is zero, the other
    rows of its key tile large: the output is the sum of the small softmax
    weights, which must keep their bits, for one and two query tiles a wave and
    with the keys in one chunk and in many.  Logits within 2e-5 of their size
    of the oracle's f32 attention (f32 sums over some hundred keys have about
    1e-6; f16 weights without a factor had 2e-3 to 4e-3 at 12 nats)."""
    cfg = cw.make_config(1, 256, n_heads, n_kv, 128, 512, 500, 460, cw.CW_F16, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 87)
    prompt = cw.synth_tokens(cw.synth_key(87, f"s{start}x{P}"), P, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    m.set_taps(True)
    m.prefill(prompt, start_pos=start)
    q = m.tap("q", 0).reshape(n_kv, n_heads // n_kv, 128).astype(np.float64)
    rng = np.random.default_rng(87)
    for nats in (12.0, 14.0, 16.0):
        k = (0.1 * rng.standard_normal((1, start, n_kv, 128))).astype(np.float16)
        v = np.zeros((1, start, n_kv, 128), np.float16)
        v[0, 1:60] = rng.uniform(-6e4, 6e4, (59, n_kv, 128))
        for g in range(n_kv):  # the shortest key that gives all of its heads the score
            k[0, 0, g] = np.linalg.lstsq(q[g], np.full(n_heads // n_kv, nats * 128 ** 0.5),
                                         rcond=None)[0]
        bits = [x.reshape(1, start, -1).view(np.uint16) for x in (k, v)]
        m.prefill_kv(*bits, start)
        m.prefill(prompt, start_pos=start)
        o = orc.OracleModel(cfg, weights)
        o.prefill_kv(*bits, start)
        ref = oracle_prompt_logits(o, prompt, start)
        o.close()
        err = float(np.max(np.abs(m.logits() - ref)) / np.max(np.abs(ref)))
        assert err <= 2e-5, (nats, err)
    m.close()


@pytest.mark.parametrize("kv", [cw.CW_F16, cw.CW_F32])
@pytest.mark.parametrize("P,start", [(1, 0), (3, 0), (4, 0), (37, 0), (5, 20)])
def test_generate_batches_its_prompt(ctx, kv, P, start):
    """generate's ids are the oracle's for prompts below and above the length
    that goes through the batched prompt phase, alone and behind a cache, and
    for a single new token; the state it leaves decodes on."""
    cfg = cw.make_config(2, 256, 4, 2, 128, 512, 1000, 96, kv, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 86)
    prompt = cw.synth_tokens(cw.synth_key(86, f"p{P}"), P + start, cfg.vocab)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    o = orc.OracleModel(cfg, weights)
    ref, _ = o.generate(prompt, 9)
    for new in (1, 7):
        if start:
            m.prefill(prompt[:start])
        toks = m.generate(prompt[start:], new, start_pos=start)
        assert np.array_equal(toks, ref[:new]), (new, toks, ref)
        assert np.array_equal(m.tokens(16), ref[:new])
        assert m.decode_next() == int(ref[new])
    m.close()
    o.close()


def test_prefill_rows_past_the_prompt_do_not_reach_it(ctx):
    """Stale rows behind the prompt (NaN) leave the logits' bits unchanged."""
    for kv, es in ((cw.CW_F16, np.float16), (cw.CW_F32, np.float32)):
        cfg = cw.make_config(1, 256, 4, 2, 128, 512, 500, 256, kv, 1e-6, 1e6)
        weights = cw.synthetic_weights(cfg, 85)
        prompt = cw.synth_tokens(cw.synth_key(85, "p"), 37, cfg.vocab)
        out = []
        for fill in (0.0, np.nan):
            m = cw.Model(ctx, cfg)
            m.set_weights(weights)
            m.finalize()
            rows = np.full((1, 256, 256), fill, es)
            bits = rows.view(np.uint16) if es is np.float16 else rows
            m.prefill_kv(bits, bits, 256)
            m.prefill(prompt)
            out.append(m.logits())
            m.close()
        assert np.array_equal(out[0], out[1])


def test_prefill_other_head_sizes_run_per_token(ctx):
    """Head sizes other than 128 (here 16, with an f32 cache) take the per-token
    step for the prompt: same logits as the oracle's loop."""
    cfg = cw.make_config(2, 64, 4, 2, 16, 128, 256, 20, cw.CW_F32, 1e-6, 1e6)
    weights = cw.synthetic_weights(cfg, 79)
    prompt = np.array([3, 1, 4, 1, 5, 9, 2, 6], np.uint32)
    m = cw.Model(ctx, cfg)
    m.set_weights(weights)
    m.finalize()
    o = orc.OracleModel(cfg, weights)
    nxt = m.prefill(prompt)
    ref_logits = oracle_prompt_logits(o, prompt)
    assert float(np.max(np.abs(m.logits() - ref_logits))) <= LOGIT_TOL
    assert nxt == int(np.argmax(ref_logits))
    m.close()
    o.close()
