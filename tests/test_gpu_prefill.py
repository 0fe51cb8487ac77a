"""A prompt read on the device a pass at a time: Session::forward(&[u32])
(crates/llm/src/model/mod.rs:842; CpuSession :1149-1158) over
forward_batch (mod.rs:544-549) = embedding rows, run_rows with
Rows::Following (llama.rs:224-289) and the head over the last row
(llama.rs:404-411); Session::prefill_pass (mod.rs:866, :1181-1183) and
CpuSession::reading (mod.rs:1079-1082); through the C ABI.

The reference's own case (crates/llm/tests/batched_decode.rs:261-290): a
23-token prompt read five tokens a pass, with the passes cut where
prefill_pass says, gives the logits of the prompt read in one call to the
bit, the same cache length, and the same next-token logits.  Beyond it:

  * logits after the prompt against the oracle's forward, token at a time
    (the reference's x86 matmul is row-by-row qrow, so a pass and m single
    steps are the same arithmetic there), at the session bar 2e-3 x max, with
    the next token the argmax of those logits exactly; passes on the
    multi-token GEMV (<= 64 rows) and on the int8 GEMM (> 64 rows), f32
    weights on the f32 GEMM;
    the attention on the pass kernel (every row's whole sequence in one
    workgroup, the default; its positions dealt over 1, 2, 4 or 8 waves,
    KVAD_PASS_WAVES) and, with KVAD_PASS_ATTN=0, on the rows launch as
    one split and as split + merged; a prompt past the single-split line
    (300 positions) both ways;
  * every stage of every layer of a pass on the device's own inputs, through
    kh_debug_llm_trace_pass, at the stage bars of test_gpu_llm_stages
    (projections 1e-5, the pushed keys 1e-6 and values exact, attention of
    row i over len + i + 1 positions 1e-5, residuals 1e-5 + half an ulp);
  * decode after a prompt: the captured steps continue from the pass's state;
  * refusals: tokens out of range and prompts past n_ctx leave the session
    as it was; an empty prompt does nothing.
"""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

import kvad_amd as K  # noqa: E402

from test_gpu_gemv import say  # noqa: E402
from test_gpu_llm import LOGIT_RTOL, build  # noqa: E402
from test_gpu_llm_stages import close_residual, proj as proj_q8  # noqa: E402
from test_gpu_moe_stages import close  # noqa: E402


def proj(w, rows, cols, x, bias=None):
    """y = x W^T (+ bias) of one row: q8 in f64 over exact block dots, q4 and
    Q4_K as the oracle's matmul gives it."""
    if not isinstance(w[0], str):
        return proj_q8(w, rows, cols, x, bias)
    x = np.ascontiguousarray(x, np.float32)
    return O.matmul_q4k(w[1], rows, cols, x, 1, bias) if w[0] == "q4k" else O.matmul_q4(w[1], w[2], rows, cols, x, 1, bias)


VARIANTS = {
    # batched_decode.rs:264: ("llama", F32), ("qwen3", Q8)
    "llama_f32": dict(bias=False, interleaved=True, tied=False, prec="f32"),
    "qwen3_q8": dict(bias=False, qk_norm=True, tied=False),
    "qwen2_q8": dict(bias=True),
    "llama_hd128_q8": dict(bias=False, interleaved=True, n_head=8, n_kv_head=2, head_dim=128, n_embd=256),
    "llama_q4k": dict(bias=False, interleaved=True, n_head=4, n_kv_head=2, head_dim=64, n_embd=256, n_ff=512,
                      prec="q4k"),
    "qwen2_q4": dict(bias=True, prec="q4"),
    # head layouts the pass kernel tiles differently (16 columns = rows x
    # the group's query heads): MHA (16 rows a tile), Qwen2.5-0.5B's group
    # of 7 (2 rows, 14 columns), MQA with 16 heads (1 row)
    "mha_q8": dict(bias=False, n_head=4, n_kv_head=4),
    "gqa7_q8": dict(bias=True, n_head=14, n_kv_head=2, n_embd=256),
    "mqa16_q8": dict(bias=False, n_head=16, n_kv_head=1, n_embd=256),
}

PROMPT = [(i * 7 + 3) % 512 for i in range(23)]  # batched_decode.rs:263 (VOCAB = 512 here)


def logits_close(got, want, what):
    scale = float(np.max(np.abs(want)))
    err = float(np.max(np.abs(np.asarray(got, np.float64) - want)))
    assert np.all(np.isfinite(got)), f"{what}: not finite"
    assert err <= LOGIT_RTOL * scale, f"{what}: max err {err:.3e} vs scale {scale:.3e}"
    return err / scale


@pytest.mark.parametrize("variant", list(VARIANTS))
def test_a_prompt_read_a_pass_at_a_time_is_the_prompt_read_at_once(ctx, variant):
    say("prefill passes vs once", variant)
    once, _ = build(ctx, 300, **VARIANTS[variant])
    passes, _ = build(ctx, 300, **VARIANTS[variant])
    once.reading(5)  # five tokens a pass: four whole passes and three left over
    passes.reading(5)
    want, want_next = once.forward_tokens(PROMPT)
    at, count, got, got_next = 0, 0, None, None
    while at < len(PROMPT):
        n = passes.prefill_pass(len(PROMPT) - at)
        assert 1 <= n <= len(PROMPT) - at, f"a pass of {n} with {len(PROMPT) - at} left"
        got, got_next = passes.forward_tokens(PROMPT[at:at + n])
        at += n
        count += 1
    assert count == 5, f"{variant}: the prompt was not read in passes"
    assert len(passes) == len(once) == len(PROMPT)
    np.testing.assert_array_equal(got, want, err_msg=f"{variant}: a pass at a time changed the logits")
    assert got_next == want_next
    # and the next token after it agrees too, so the caches do
    a, na = passes.forward_tokens([9])
    b, nb = once.forward_tokens([9])
    np.testing.assert_array_equal(a, b)
    assert na == nb


def test_prefill_pass_cuts_whole_chunks_from_the_front(ctx, monkeypatch):
    say("prefill_pass")
    m, _ = build(ctx, 301)
    # the default: 512 a pass, the reference's GPU backend's chunk (gpu/src/model.rs:897)
    assert [m.prefill_pass(n) for n in (1, 63, 512, 513, 2000)] == [1, 63, 512, 512, 512]
    m.reading(5)
    assert [m.prefill_pass(n) for n in (23, 5, 3, 0)] == [5, 5, 3, 0]
    m.reading(0)
    monkeypatch.setenv("KVAD_PREFILL_CHUNK", "16")
    assert m.prefill_pass(40) == 16
    with pytest.raises(K.KvadError):
        m.reading(1 << 16)


CASES = {
    # (variant, prompt length, chunk, attention: the pass kernel, or the
    # rows launch as one split or split + merged)
    "gemv_rows": ("qwen2_q8", 23, 64, "pass"),       # one pass of 23 rows: multi-token GEMVs
    "gemv_rows_single": ("qwen2_q8", 23, 64, "single"),
    "rows40_single": ("qwen2_q8", 40, 40, "single"),
    "rows40_pass": ("qwen3_q8", 40, 40, "pass"),
    "rows40_split": ("qwen3_q8", 40, 40, "split"),   # every row split and merged
    "gemm_rows": ("qwen2_q8", 70, 70, "single"),     # one pass of 70 rows: the int8 GEMM
    "gemm_pass": ("qwen3_q8", 70, 70, "pass"),
    "f32_gemm": ("llama_f32", 40, 40, "pass"),       # the f32 GEMM
    "q4k_rows": ("llama_q4k", 37, 64, "pass"),
    "q4k_gemm": ("llama_q4k", 70, 70, "pass"),
    "q4_gemm": ("qwen2_q4", 70, 70, "pass"),
    "q4_passes": ("qwen2_q4", 23, 7, "pass"),
    "hd128_passes": ("llama_hd128_q8", 30, 8, "pass"),
    "hd128_passes_w8": ("llama_hd128_q8", 30, 8, "pass:8"),
    "hd128_split": ("llama_hd128_q8", 30, 8, "split"),
    "rows40_pass_w4": ("qwen2_q8", 40, 40, "pass:4"),
}


def attention_path(monkeypatch, attn):
    # "pass" (waves per workgroup by the launch's rule), "pass:W" (W waves),
    # "single" / "split": the rows launch
    if attn.startswith("pass:"):
        monkeypatch.setenv("KVAD_PASS_WAVES", attn[5:])
    elif attn != "pass":
        monkeypatch.setenv("KVAD_PASS_ATTN", "0")
    if attn == "split":
        monkeypatch.setenv("KVAD_ATTN_SINGLE", "0")


@pytest.mark.parametrize("case", list(CASES))
def test_prefill_matches_the_oracle(ctx, monkeypatch, case):
    variant, n, chunk, attn = CASES[case]
    attention_path(monkeypatch, attn)
    say("prefill vs oracle", case)
    m, mk = build(ctx, 310, n_ctx=max(64, n + 8), **VARIANTS[variant])
    m.reading(chunk)
    ref = mk()
    prompt = [(i * 13 + 5) % 512 for i in range(n)]
    logits, nxt = m.forward_tokens(prompt)
    for t in prompt:
        want = ref.forward(t)
    worst = logits_close(logits, want, f"{case} after the prompt")
    assert nxt == O.argmax(logits), "the next token is not the argmax of the last logits"
    assert len(m) == n
    # decoding goes on from the prompt's cache
    for step, t in enumerate([nxt, 9, 400]):
        lg, nt = m.forward(int(t))
        worst = max(worst, logits_close(lg, ref.forward(int(t)), f"{case} decode step {step}"))
        assert nt == O.argmax(lg)
    say("prefill vs oracle worst", case, f"{worst:.2e}")


@pytest.mark.parametrize("attn", ["pass", "pass:8", "single"])
@pytest.mark.parametrize("chunk", [64, 512])
def test_a_prompt_past_the_single_split_line(ctx, monkeypatch, chunk, attn):
    # 300 positions at head_dim 64: passes of 64 rows, or one pass of 300
    # rows, on the pass kernel or on the rows launch (one split up to 256
    # positions, split + merged past them)
    attention_path(monkeypatch, attn)
    say("prefill past the single split", chunk, attn)
    m, mk = build(ctx, 320, n_layer=1, n_ctx=512)
    m.reading(chunk)
    ref = mk()
    prompt = [(i * 11 + 2) % 512 for i in range(300)]
    logits, nxt = m.forward_tokens(prompt)
    for t in prompt:
        want = ref.forward(t)
    logits_close(logits, want, "after 300 tokens")
    assert nxt == O.argmax(logits) and len(m) == 300


def test_generation_continues_from_the_prompt(ctx):
    say("prefill then generate")
    a, _ = build(ctx, 330)
    b, _ = build(ctx, 330)
    _, na = a.forward_tokens(PROMPT)
    _, nb = b.forward_tokens(PROMPT)
    assert na == nb
    got = a.generate(na, 8)  # the captured step from the pass's state
    t, want = nb, []
    for _ in range(8):
        _, t = b.forward(t)
        want.append(t)
    np.testing.assert_array_equal(got, want)


def test_refusals_leave_the_session_as_it_was(ctx):
    say("prefill refusals")
    m, _ = build(ctx, 340, n_ctx=32)
    plain, _ = build(ctx, 340, n_ctx=32)
    m.forward_tokens([1, 2, 3])
    plain.forward_tokens([1, 2, 3])
    with pytest.raises(K.KvadError, match="out of range"):
        m.forward_tokens([4, 512, 6])
    with pytest.raises(K.KvadError, match="overrun"):
        m.forward_tokens(list(range(30)))
    lg, nt = m.forward_tokens([])
    assert len(m) == 3
    a, na = m.forward_tokens([7, 8])
    b, nb = plain.forward_tokens([7, 8])
    np.testing.assert_array_equal(a, b)
    assert na == nb


STAGE_VARIANTS = {
    # (variant, positions held, rows in the pass, attention)
    "qwen2_gemv": ("qwen2_q8", 3, 6, "pass"),          # 3 positions held, a pass of 6 rows
    "qwen3_40": ("qwen3_q8", 2, 40, "pass"),
    "qwen3_40_rows": ("qwen3_q8", 2, 40, "single"),
    "llama_hd128": ("llama_hd128_q8", 4, 12, "pass"),
    "llama_hd128_split": ("llama_hd128_q8", 4, 12, "split"),
    "qwen2_long": ("qwen2_q8", 70, 37, "pass"),        # rows over 71 .. 107 positions
    "qwen2_long_w2": ("qwen2_q8", 70, 37, "pass:2"),   # the positions dealt over 2, 4, 8 waves
    "qwen2_long_w4": ("qwen2_q8", 70, 37, "pass:4"),
    "qwen2_long_w8": ("qwen2_q8", 70, 37, "pass:8"),
    "hd128_long_w4": ("llama_hd128_q8", 50, 21, "pass:4"),
    "mha": ("mha_q8", 5, 37, "pass"),
    "gqa7": ("gqa7_q8", 5, 37, "pass:4"),
    "mqa16": ("mqa16_q8", 5, 37, "pass:2"),
}


@pytest.mark.parametrize("case", list(STAGE_VARIANTS))
def test_each_stage_of_a_pass(ctx, monkeypatch, case):
    variant, held, n, attn = STAGE_VARIANTS[case]
    attention_path(monkeypatch, attn)
    stages(ctx, case, held, n, 3, VARIANTS[variant])


GEMM_STAGES = {
    # (layers, tokens per tile, or None: the rule's; sizes).  q/k/v and gate/up
    # each in one launch of weights of unequal rows: 384 and 192 (a tile and a
    # half of 128 rows), and 1568 (no multiple of any tile)
    "q8": (2, None, dict(bias=True)),
    "q8_128": (2, "128", dict(bias=True, n_head=6, n_kv_head=3, n_ff=1568)),
    "q8_split": (1, None, dict(bias=True, n_head=6, n_kv_head=3, n_embd=1568, n_ff=1568)),
    "q8_split_128": (1, "128", dict(bias=True, n_head=6, n_kv_head=3, n_embd=1568, n_ff=1568)),
    "q4": (2, None, dict(bias=True, prec="q4")),
    "q4_split_32": (1, "32", dict(bias=True, prec="q4", n_head=6, n_kv_head=3, n_embd=1568, n_ff=1568)),
    "q4k": (2, None, dict(bias=True, prec="q4k", n_embd=256, n_ff=512)),
    "q4k_split": (1, None, dict(bias=True, prec="q4k", n_head=8, n_kv_head=2, n_embd=1536, n_ff=1536)),
    "q4k_split_64": (1, "64", dict(bias=True, prec="q4k", n_head=4, n_kv_head=1, n_embd=1536, n_ff=1536)),
}


@pytest.mark.parametrize("case", list(GEMM_STAGES))
def test_each_stage_of_a_pass_on_the_gemm(ctx, monkeypatch, case):
    # 67 rows: past the multi-token GEMV; twelve k-stages and more are split
    # over the grid, the weights' partials one behind the other
    n_layer, tile, kw = GEMM_STAGES[case]
    if tile:
        monkeypatch.setenv("KVAD_GEMM_TILE_M", tile)
    stages(ctx, case, 2, 67, n_layer, kw, ties=True)


def tie_slack(h):
    """What a product with h may move by where the device's own rounding of h
    (the norm's sum, swiglu's exponential: a few ulps, under 1e-4 of a code)
    decides between two codes: a step of each such code times the largest
    weight (normal, 0.02: under 0.12; a tied head's 0.5, 25 times that).  One in
    5000 values lies so near."""
    b = np.abs(np.asarray(h, np.float64)).reshape(-1, 32)
    step = b.max(1, keepdims=True) / 127
    t = b / np.maximum(step, 1e-30)
    return 0.12 * float((step * (np.abs(t - np.floor(t) - 0.5) < 1e-4)).sum())


def stages(ctx, case, held, n, n_layer, kw, ties=False):
    slack = tie_slack if ties else lambda h: 0.0
    near = lambda got, want, what, h: close(got, want, what, rtol=1e-5 + slack(h) / float(np.max(np.abs(want))))
    say("prefill stages", case)
    m, mk = build(ctx, 350, n_layer=n_layer, n_ctx=max(64, held + n), **kw)
    m.reading(n)
    ref = mk()  # for its weights, norms and tables only
    s = ref.s
    e, hd, nh, nkv, eps = s["n_embd"], s["head_dim"], s["n_head"], s["n_kv_head"], s["eps"]
    qd, kvd, half, ff = nh * hd, nkv * hd, hd // 2, s["n_ff"]
    rope = O.rope_apply_interleaved if s.get("rope_interleaved") else O.rope_apply
    if held:
        m.forward_tokens([(i * 5 + 1) % 512 for i in range(held)])
    toks = [(i * 17 + 4) % 512 for i in range(n)]
    tr = m.trace_pass(toks)
    assert len(m) == held + n
    worst = {}
    note = lambda name, r: worst.__setitem__(name, max(worst.get(name, 0.0), r))
    for i, t in enumerate(toks):
        np.testing.assert_array_equal(tr["x_embed"][i], O.row_q8(*ref.embed, e, t), err_msg=f"embedding row {i}")
    X = tr["x_embed"]
    for l, L in enumerate(ref.layers):
        X_attn, X_mlp = tr["x_attn"][l], tr["x_mlp"][l]
        kc, vc = tr["k_cache"][l], tr["v_cache"][l]
        for i in range(n):
            pos, where = held + i, f"layer {l} row {i}"
            x = X[i]
            h = O.rms_norm(x, L["attn_norm"], eps)
            qkv = tr["qkv"][l][i]
            note("q", near(qkv[:qd], proj(L["q"], qd, e, h, L.get("q_b")), f"{where} q", h))
            note("k", near(qkv[qd:qd + kvd], proj(L["k"], kvd, e, h, L.get("k_b")), f"{where} k", h))
            note("v", near(qkv[qd + kvd:], proj(L["v"], kvd, e, h, L.get("v_b")), f"{where} v", h))
            q, k = qkv[:qd].copy(), qkv[qd:qd + kvd].copy()
            for head in range(nkv):
                seg = k[head * hd:(head + 1) * hd]
                if L.get("k_norm") is not None:
                    seg = O.rms_norm(seg, L["k_norm"], eps)
                k[head * hd:(head + 1) * hd] = rope(ref.cos, ref.sin, half, seg, pos)
            for head in range(nh):
                seg = q[head * hd:(head + 1) * hd]
                if L.get("q_norm") is not None:
                    seg = O.rms_norm(seg, L["q_norm"], eps)
                q[head * hd:(head + 1) * hd] = rope(ref.cos, ref.sin, half, seg, pos)
            note("k push", close(kc[pos], k, f"{where} k push", rtol=1e-6))
            np.testing.assert_array_equal(vc[pos], qkv[qd + kvd:], err_msg=f"{where} v push")
            # row i attends over the held positions and the pass's rows up to itself
            att = O.attend(nh, nkv, hd, q, kc[:pos + 1].ravel(), vc[:pos + 1].ravel(), pos + 1)
            note("attention", close(tr["att"][l][i], att, f"{where} attention"))
            y = proj(L["o"], e, qd, tr["att"][l][i])
            note("o + x", close_residual(X_attn[i], x, y, f"{where} o + residual"))
            h = O.rms_norm(X_attn[i], L["mlp_norm"], eps)
            note("gate", near(tr["gate"][l][i], proj(L["gate"], ff, e, h), f"{where} gate", h))
            note("up", near(tr["up"][l][i], proj(L["up"], ff, e, h), f"{where} up", h))
            g = O.swiglu(tr["gate"][l][i], tr["up"][l][i])
            y = proj(L["down"], e, ff, g)
            note("down + x", close_residual(X_mlp[i], X_attn[i], y, f"{where} down + residual", slack(g)))
        X = X_mlp
    h = O.rms_norm(X[n - 1], ref.final_norm, eps)
    logits = proj(ref.head, s["vocab"], e, h)
    note("head", close(tr["logits"], logits, "head of the last row", rtol=1e-5 + 25 * slack(h) / float(np.max(np.abs(logits)))))
    say("prefill stages worst", case, {k: f"{v:.1e}" for k, v in worst.items()})


@pytest.mark.parametrize("variant,attn", [("qwen3_q8", "pass"), ("qwen3_q8", "pass:4"), ("qwen3_q8", "pass:8"),
                                          ("qwen3_hd128_q8", "pass:2")])
@pytest.mark.parametrize("spread", [1.0, 2.5, 6.0])
def test_a_pass_over_widely_spread_scores(ctx, monkeypatch, variant, attn, spread):
    # The query norms scaled so that scores spread by about `spread`: by 2.5 a
    # later tile's maximum passes the first's by more than 8 now and then (the
    # running sums are rescaled), by 6 weights fall under 1e-8 as well and the
    # workgroup drops them as the reference does, in a second pass.
    kw = dict(VARIANTS["qwen3_q8"], **({"n_head": 8, "n_kv_head": 2, "head_dim": 128, "n_embd": 256}
                                       if variant == "qwen3_hd128_q8" else {}))
    attention_path(monkeypatch, attn)
    say("pass, spread scores", variant, attn, spread)
    n = 150
    m, mk = build(ctx, 360, n_layer=1, n_ctx=192, **kw)
    ref = mk()
    s, L = ref.s, ref.layers[0]
    hd, nh, nkv, half, eps = s["head_dim"], s["n_head"], s["n_kv_head"], s["head_dim"] // 2, s["eps"]
    qd, kvd = nh * hd, nkv * hd
    L["q_norm"] = (np.asarray(L["q_norm"]) * spread).astype(np.float32)
    m.set_layer(0, *m._keep[0], L["attn_norm"], L["mlp_norm"], L.get("q_b"), L.get("k_b"), L.get("v_b"), L["q_norm"],
                L["k_norm"])
    tr = m.trace_pass([(i * 29 + 7) % 512 for i in range(n)])
    kc, vc, dropped = tr["k_cache"][0], tr["v_cache"][0], 0
    for i in range(n):
        q = tr["qkv"][0][i][:qd].copy()
        for head in range(nh):
            seg = O.rms_norm(q[head * hd:(head + 1) * hd], L["q_norm"], eps)
            rope = O.rope_apply_interleaved if s.get("rope_interleaved") else O.rope_apply
            q[head * hd:(head + 1) * hd] = rope(ref.cos, ref.sin, half, seg, i)
            sc = kc[:i + 1].reshape(i + 1, nkv, hd)[:, head // (nh // nkv)] @ q[head * hd:(head + 1) * hd] / np.sqrt(hd)
            dropped += int(np.sum(np.exp(sc - sc.max()) / np.sum(np.exp(sc - sc.max())) < 1e-8))
        att = O.attend(nh, nkv, hd, q, kc[:i + 1].ravel(), vc[:i + 1].ravel(), i + 1)
        close(tr["att"][0][i], att, f"row {i} attention")
    assert dropped == 0 if spread == 1.0 else spread < 6.0 or dropped > 0, dropped


@pytest.mark.parametrize("attn", ["pass:1", "pass:2", "pass:8"])
@pytest.mark.parametrize("spread,even", [(2.2, 0), (4.0, 0), (4.0, 270), (4.0, 150)])
def test_a_pass_that_drops_weights_it_foresees_or_finds(ctx, monkeypatch, attn, spread, even):
    # 300 rows, up to nineteen 16-position tiles a wave: weights under 1e-8 in
    # sight from the first tile on (4.0), now and then or only at the end
    # (2.2), or not before the first `even` positions, one token repeated, are
    # over.  The pass gives the same bits every time, whichever wave tells the
    # others first.
    monkeypatch.setenv("KVAD_PASS_WAVES", attn[5:])
    say("pass, dropped weights", attn, spread, even)
    n = 300
    m, mk = build(ctx, 370, n_layer=1, n_ctx=320, **VARIANTS["qwen3_q8"])
    ref = mk()
    s, L = ref.s, ref.layers[0]
    hd, nh, nkv, half, eps = s["head_dim"], s["n_head"], s["n_kv_head"], s["head_dim"] // 2, s["eps"]
    qd = nh * hd
    L["q_norm"] = (np.asarray(L["q_norm"]) * spread).astype(np.float32)
    m.set_layer(0, *m._keep[0], L["attn_norm"], L["mlp_norm"], L.get("q_b"), L.get("k_b"), L.get("v_b"), L["q_norm"],
                L["k_norm"])
    m.reading(n)
    toks = [11 if i < even else (i * 29 + 7) % 512 for i in range(n)]
    tr = m.trace_pass(toks)
    kc, vc, dropped = tr["k_cache"][0], tr["v_cache"][0], 0
    for i in range(0, n, 7):
        q = tr["qkv"][0][i][:qd].copy()
        for head in range(nh):
            seg = O.rms_norm(q[head * hd:(head + 1) * hd], L["q_norm"], eps)
            q[head * hd:(head + 1) * hd] = O.rope_apply(ref.cos, ref.sin, half, seg, i)
            sc = kc[:i + 1].reshape(i + 1, nkv, hd)[:, head // (nh // nkv)] @ q[head * hd:(head + 1) * hd] / np.sqrt(hd)
            dropped += int(np.sum(np.exp(sc - sc.max()) / np.sum(np.exp(sc - sc.max())) < 1e-8))
        att = O.attend(nh, nkv, hd, q, kc[:i + 1].ravel(), vc[:i + 1].ravel(), i + 1)
        close(tr["att"][0][i], att, f"row {i} attention")
    assert dropped > 0 or spread < 4.0, dropped
    for _ in range(3):
        m.truncate(0)
        np.testing.assert_array_equal(m.trace_pass(toks)["att"], tr["att"])


def test_widely_spread_scores_cost_a_second_pass_at_most(ctx):
    # Where most workgroups drop some weight (scores spread by 4 over 6000
    # positions) the attention goes over the positions twice, 1.6 times one
    # pass's time, and a prompt of one layer takes 1.3 times as long; found
    # only at the end and gone over twice more, 2.6 and 1.8.
    import time

    say("pass, time of spread scores")
    n = 6000
    m, mk = build(ctx, 380, n_layer=1, n_ctx=n, **dict(VARIANTS["qwen3_q8"], n_head=14, n_kv_head=2, n_embd=128))
    ref = mk()
    L = ref.layers[0]
    toks = np.random.default_rng(3).integers(0, 512, n).astype(np.int32)
    best = {}
    for spread in (0.5, 4.0):
        m.set_layer(0, *m._keep[0], L["attn_norm"], L["mlp_norm"], L.get("q_b"), L.get("k_b"), L.get("v_b"),
                    (np.asarray(L["q_norm"]) * spread).astype(np.float32), L["k_norm"])
        times = []
        for _ in range(8):
            m.truncate(0)
            t = time.perf_counter()
            m.forward_tokens(toks)
            times.append(time.perf_counter() - t)
        best[spread] = min(times)
    say("pass, time of spread scores, ms", {k: round(1e3 * v, 2) for k, v in best.items()})
    assert best[4.0] <= 1.55 * best[0.5], best


@pytest.mark.parametrize("prec,n_embd,n,multi", [("q8", 4128, 40, False), ("q4", 4128, 17, False), ("q4k", 4352, 49, False),
                                                 ("q8", 4128, 16, True), ("q8", 4096, 40, True), ("q4k", 4352, 48, True)])
def test_joint_projections_of_wide_rows(ctx, monkeypatch, prec, n_embd, n, multi):
    # q/k/v of one pass past 16 rows: on the GEMM where the multi-token GEMV,
    # which cannot split several weights over the grid, would stream them once
    # per 16 rows.  The GEMM's sums of a row (its k-stages unsplit) do not
    # depend on the rows beside it: bit for bit those of 70 rows, which always
    # take it; the GEMV's run in another order.
    monkeypatch.setenv("KVAD_GEMM_KSPLIT", "1")
    say("joint projections", prec, n_embd, n)
    m, mk = build(ctx, 390, n_layer=1, n_ctx=96, n_embd=n_embd, n_head=4, n_kv_head=1, head_dim=64, n_ff=256, prec=prec)
    m.reading(70)
    ref = mk()
    s, L = ref.s, ref.layers[0]
    toks = [(i * 19 + 6) % 512 for i in range(70)]
    few = m.trace_pass(toks[:n])
    m.truncate(0)
    many = m.trace_pass(toks)["qkv"][0][:n]
    same = np.array_equal(few["qkv"][0], many)
    assert same != multi
    qd, kvd = 256, 64
    for i in (0, n // 2, n - 1):
        h = O.rms_norm(few["x_embed"][i], L["attn_norm"], s["eps"])
        for at, name, rows in ((0, "q", qd), (qd, "k", kvd), (qd + kvd, "v", kvd)):
            want = proj(L[name], rows, n_embd, h, L.get(name + "_b"))
            for got in (few["qkv"][0], many):
                close(got[i, at:at + rows], want, f"row {i} {name}")
