"""The attention entry point that allocates nothing (kh_attend_dev_noalloc):
its output equals kh_attend_dev's, bit for bit, on two calls in a row, the
second with a smaller input; a call whose partials exceed the library's
static scratch array is refused with a clear error.  And calls that need no
scratch of their context, captured into a graph on one that has made none."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

import kvad_amd as K  # noqa: E402


def say(*a):
    print("[case]", *a, flush=True)


def run(ctx, fn, n_head, n_kv, hd, q, k, v, L, out):
    rc = fn(ctx.h, n_head, n_kv, hd, q.data_ptr(), k.data_ptr(), v.data_ptr(), L, out.data_ptr())
    return rc


@pytest.mark.parametrize("geom,lengths", [((14, 2, 64), (8192, 1000)), ((32, 8, 128), (4096, 300)),
                                          ((14, 2, 64), (32768, 1))])
def test_noalloc_attention_equals_the_allocating_entry(ctx, geom, lengths):
    import torch

    n_head, n_kv, hd = geom
    kv_dim = n_kv * hd
    g = torch.Generator(device="cuda")
    g.manual_seed(1234)
    Lmax = max(lengths)
    k = torch.randn(Lmax, kv_dim, device="cuda", generator=g)
    v = torch.randn(Lmax, kv_dim, device="cuda", generator=g)
    for L in lengths:  # the second call is smaller than the first
        say("noalloc", geom, L)
        q = torch.randn(n_head * hd, device="cuda", generator=g)
        want = torch.empty(n_head * hd, device="cuda")
        got = torch.full((n_head * hd,), float("nan"), device="cuda")
        torch.cuda.synchronize()
        assert run(ctx, K.lib.kh_attend_dev, n_head, n_kv, hd, q, k, v, L, want) == 0, K.lib.kh_last_error()
        assert run(ctx, K.lib.kh_attend_dev_noalloc, n_head, n_kv, hd, q, k, v, L, got) == 0, K.lib.kh_last_error()
        ctx.synchronize()
        np.testing.assert_array_equal(got.cpu().numpy(), want.cpu().numpy())


def test_noalloc_attention_of_no_positions_is_zero(ctx):
    import torch

    say("noalloc L=0")
    q = torch.randn(14 * 64, device="cuda")
    out = torch.full((14 * 64,), 7.0, device="cuda")
    torch.cuda.synchronize()
    assert K.lib.kh_attend_dev_noalloc(ctx.h, 14, 2, 64, q.data_ptr(), None, None, 0, out.data_ptr()) == 0
    ctx.synchronize()
    assert not out.cpu().numpy().any()


def test_noalloc_attention_refuses_what_exceeds_the_scratch(ctx):
    import torch

    assert K.lib.kh_noalloc_scratch_bytes() == 8 << 20
    # 64 heads of 128 over 32768 positions: 128 splits x 64 heads of partials (12.7 MB)
    n_head, n_kv, hd, L = 64, 8, 128, 32768
    say("noalloc too large", n_head, L)
    k = torch.zeros(L, n_kv * hd, device="cuda")
    v = torch.zeros(L, n_kv * hd, device="cuda")
    q = torch.zeros(n_head * hd, device="cuda")
    out = torch.empty(n_head * hd, device="cuda")
    torch.cuda.synchronize()
    rc = run(ctx, K.lib.kh_attend_dev_noalloc, n_head, n_kv, hd, q, k, v, L, out)
    assert rc == -1  # KH_EINVAL
    assert b"bytes of scratch" in K.lib.kh_last_error()


def captured(ctx, call):
    """The call captured into a graph on a stream of its own, on a context
    that has made no scratch yet."""
    import torch

    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=stream):
        call()
    return g, stream


def replays_match(ctx, g, stream, out, want, tol):
    """Several replays, the context's own eager work between them: a matmul
    whose scratch grows past what was there, so that whatever the graph still
    named would have moved."""
    import torch

    for i in range(4):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            g.replay()
        torch.cuda.synchronize()
        err = float((out - want).abs().max())
        assert err <= tol * float(want.abs().max()), (i, err)
        x = torch.randn((1 << i) * 500, 2048, device="cuda")
        d, y = torch.randn(64, 2048, device="cuda"), torch.empty(x.shape[0], 64, device="cuda")
        torch.cuda.synchronize()
        w = K.Weight.quantize_dev(ctx, 64, 2048, d.data_ptr(), K.Q8)
        w.matmul_bt_dev(x.data_ptr(), x.shape[0], y.data_ptr())
        ctx.synchronize()


@pytest.mark.parametrize("L", [20, 33, 64])
def test_latent_attention_of_one_launch_is_captured_without_scratch(ctx, L):
    import torch

    say("mla under capture", L)
    H = 16
    g = torch.Generator(device="cuda")
    g.manual_seed(L)
    ql, qp, c, pe = (torch.randn(*s, device="cuda", generator=g) for s in ((H, 512), (H, 64), (L, 512), (L, 64)))
    want, out = torch.empty(H, 512, device="cuda"), torch.empty(H, 512, device="cuda")

    def call(cx, o):
        K.mla_attend_dev(cx, H, ql.data_ptr(), qp.data_ptr(), c.data_ptr(), pe.data_ptr(), L, 192.0 ** -0.5, o.data_ptr())

    torch.cuda.synchronize()
    call(ctx, want)
    ctx.synchronize()
    fresh = K.Context(0)
    try:
        graph, stream = captured(fresh, lambda: call(fresh, out))
        replays_match(fresh, graph, stream, out, want, 1e-5)
    finally:
        fresh.set_stream(None)
        fresh.close()


@pytest.mark.parametrize("prec,m,rows,cols", [("q8", 2, 65536, 256), ("q8", 3, 8960, 1536), ("q4", 4, 4096, 3072)])
def test_few_rows_are_captured_without_scratch(ctx, prec, m, rows, cols):
    import torch

    say("matmul under capture", prec, m, rows, cols)
    g = torch.Generator(device="cuda")
    g.manual_seed(rows)
    data = torch.randn(rows, cols, device="cuda", generator=g) * 0.02
    x = torch.randn(m, cols, device="cuda", generator=g)
    want, out = torch.empty(m, rows, device="cuda"), torch.empty(m, rows, device="cuda")
    torch.cuda.synchronize()
    fresh = K.Context(0)
    try:
        for cx, o in ((ctx, want), (fresh, out)):
            w = K.Weight.quantize_dev(cx, rows, cols, data.data_ptr(), K.Q8 if prec == "q8" else K.Q4)
            cx.synchronize()
            call = lambda: w.matmul_bt_dev(x.data_ptr(), m, o.data_ptr())  # noqa: E731
            if cx is ctx:
                call()
                cx.synchronize()
        graph, stream = captured(fresh, call)
        replays_match(fresh, graph, stream, out, want, 1e-5)
    finally:
        fresh.set_stream(None)
        fresh.close()
