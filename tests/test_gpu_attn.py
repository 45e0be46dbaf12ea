"""GPU parity of the gated full-attention core (qw_attn_forward) against the
CPU oracle (orc_full_attn_seq, pinned bit-exactly to the reference's own
FullAttention::forward in tests/test_oracle.py).

Shapes: Qwen3.5-0.8B full attention, 8 query heads, 2 KV heads, head dim 256,
rotary 64 dims, theta 1e7 (also head dim 128 and theta 100 for large angles).
Sequences are prefilled and then decoded through the GPU cache; the oracle
runs the same token stream through its own cache.

Bars (normwise relative error against the oracle):
  FP32 cache, FP32 io      2e-5: only reduction orders (norms, dot products,
                           online softmax), __expf and the device cosf/sinf
                           differ; measured ~1e-6.
  INT8 cache               5e-3: the same, plus f16 MFMA operands for q and
                           p (2^-11; measured ~2.5e-4), plus INT8
                           rounding flips where the
                           GPU's and the oracle's normalized k or v land on
                           either side of a .5 step (one step = 1/127 of the
                           head's max); the cached codes are checked to differ
                           by at most one step, on at most 1% of entries.
  BF16 io                  1e-2: inputs rounded identically for both sides; the
                           output carries one BF16 rounding.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

NH, NKV, HD, ROT = 8, 2, 256, 64


def dev(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").to(dtype)


def host(t):
    return t.float().cpu().numpy()


class Stream:
    """B sequences of raw projections, one stacked row per token:
    [q0 g0 q1 g1 ... q7 g7 | k | v] (the interleaved Q|gate projection output)."""

    def __init__(self, oracle, B, T, seed, hd=HD, nh=NH, nkv=NKV):
        self.hd, self.nh, self.nkv = hd, nh, nkv
        self.ld = nh * 2 * hd + 2 * nkv * hd
        self.rows = oracle.normal((B, T, self.ld), seed)
        self.qn = oracle.normal((hd,), seed + 1, 0.0, 0.1)
        self.kn = oracle.normal((hd,), seed + 2, 0.0, 0.1)

    def parts(self, rows):
        """(q, gate, k, v) numpy arrays of rows [..., ld] for the oracle."""
        nh, hd, nkv = self.nh, self.hd, self.nkv
        qg = rows[..., :nh * 2 * hd].reshape(rows.shape[:-1] + (nh, 2, hd))
        q = qg[..., 0, :].reshape(rows.shape[:-1] + (nh * hd,))
        g = qg[..., 1, :].reshape(rows.shape[:-1] + (nh * hd,))
        k = rows[..., nh * 2 * hd:nh * 2 * hd + nkv * hd]
        v = rows[..., nh * 2 * hd + nkv * hd:]
        return [np.ascontiguousarray(x) for x in (q, g, k, v)]

    def views(self, drows):
        """(q, gate, k, v) device views of rows [R, ld]: q at head stride 2*hd."""
        nh, hd, nkv = self.nh, self.hd, self.nkv
        return drows[:, 0:], drows[:, hd:], drows[:, nh * 2 * hd:], drows[:, nh * 2 * hd + nkv * hd:]


def run_gpu(qw, ctx, st, cache, drows, pos, tokens, theta, rot, out_dtype=torch.float32, max_len=0):
    q, g, k, v = st.views(drows)
    out = torch.empty(drows.shape[0], st.nh * st.hd, device="cuda", dtype=out_dtype)
    qw.attn_forward(ctx, dev(st.qn), dev(st.kn), cache, dev(np.array(pos, np.int32), torch.int32), q, g, k, v, out,
                    num_heads=st.nh, num_kv_heads=st.nkv, head_dim=st.hd, rotary_dim=rot, rope_theta=theta,
                    tokens=tokens, q_head_stride=2 * st.hd, max_len=max_len)
    return out


def oracle_stream(oracle, st, rows_b, int8, theta, rot, capacity):
    """All tokens of one sequence through the oracle (its own cache)."""
    q, g, k, v = st.parts(rows_b)
    out, cache = oracle.full_attn_seq(q, g, k, v, st.qn, st.kn, st.nh, st.nkv, st.hd, rotary_dim=rot, theta=theta,
                                      int8=int8, capacity=capacity)
    return out, cache


@pytest.mark.parametrize("int8,io,hd,theta", [(False, "f32", 256, 1.0e7), (True, "f32", 256, 1.0e7),
                                              (True, "bf16", 256, 1.0e7), (False, "f32", 128, 100.0),
                                              (True, "f32", 128, 100.0)])
def test_attn_prefill_then_decode(qw, ctx, oracle, relerr, int8, io, hd, theta):
    """3 sequences: a 37-token prefill (one launch over all 111 rows, causal
    within each sequence), then 5 decode steps of one token each."""
    B, T0, steps, cap = 3, 37, 5, 64
    rot = hd // 4
    st = Stream(oracle, B, T0 + steps, 200 + hd + int(int8), hd=hd)
    tdt = torch.float32 if io == "f32" else torch.bfloat16
    rows = st.rows if io == "f32" else host(dev(st.rows, torch.bfloat16))  # what the GPU sees
    cache = qw.kv_cache(B, cap, st.nkv, hd, int8=int8)
    outs = [run_gpu(qw, ctx, st, cache, dev(st.rows[:, :T0].reshape(B * T0, -1), tdt), [0] * B, T0, theta, rot,
                    out_dtype=tdt)]
    for s in range(steps):
        outs.append(run_gpu(qw, ctx, st, cache, dev(st.rows[:, T0 + s], tdt), [T0 + s] * B, 1, theta, rot,
                            out_dtype=tdt))
    torch.cuda.synchronize()
    got = np.concatenate([host(outs[0]).reshape(B, T0, -1)] + [host(o)[:, None] for o in outs[1:]], axis=1)
    bar = (5e-3 if int8 else 2e-5) if io == "f32" else 1e-2
    for b in range(B):
        ref, (kc, vc, ks, vs) = oracle_stream(oracle, st, rows[b], int8, theta, rot, cap)
        err = relerr(got[b], ref)
        print("attn", int8, io, hd, b, err)
        assert err <= bar, (b, err)
        gk, gv = host(cache[0][b]), host(cache[1][b])
        n = T0 + steps
        if int8:
            for gc, oc in ((gk, kc), (gv, vc)):
                d = np.abs(gc[:n].astype(np.int32) - oc[:n].astype(np.int32))
                assert d.max() <= 1 and (d > 0).mean() <= 0.01, (d.max(), (d > 0).mean())
            np.testing.assert_allclose(host(cache[2][b])[:n], ks[:n], rtol=2e-5)
            np.testing.assert_allclose(host(cache[3][b])[:n], vs[:n], rtol=2e-5)
        else:
            assert relerr(gk[:n], kc[:n]) <= 2e-5 and relerr(gv[:n], vc[:n]) <= 2e-5


def test_attn_ragged_positions(qw, ctx, oracle, relerr):
    """Sequences at different positions in one decode launch: each attends to
    exactly its own prefix (positions 0, 9 and 30)."""
    B, cap = 3, 48
    lens = [1, 10, 31]
    st = Stream(oracle, B, max(lens), 300)
    cache = qw.kv_cache(B, cap, int8=False)
    # prefill each sequence to lens[b]-1 tokens with its own launch, then one decode step for all
    for b in range(B):
        n = lens[b] - 1
        if n:
            sub = tuple(c[b:b + 1] for c in cache)
            run_gpu(qw, ctx, st, sub, dev(st.rows[b, :n]), [0], n, 1.0e7, ROT)
    out = run_gpu(qw, ctx, st, cache, dev(np.stack([st.rows[b, lens[b] - 1] for b in range(B)])),
                  [n - 1 for n in lens], 1, 1.0e7, ROT)
    torch.cuda.synchronize()
    for b in range(B):
        ref, _ = oracle_stream(oracle, st, st.rows[b, :lens[b]], False, 1.0e7, ROT, cap)
        assert relerr(host(out)[b], ref[-1]) <= 2e-5


@pytest.mark.parametrize("int8", [False, True])
def test_attn_long_context_decode(qw, ctx, oracle, relerr, int8):
    """A 3000-token cache built by one GPU prefill, then a decode step split
    over many key ranges: checked against the oracle's attention over the
    GPU-written cache (dequantized with its own scales) and the oracle's
    norm + RoPE of the new token."""
    L, cap = 3000, 3072
    st = Stream(oracle, 1, L + 1, 400)
    cache = qw.kv_cache(1, cap, int8=int8)
    run_gpu(qw, ctx, st, cache, dev(st.rows[0, :L]), [0], L, 1.0e7, ROT)
    out = run_gpu(qw, ctx, st, cache, dev(st.rows[0, L:L + 1]), [L], 1, 1.0e7, ROT)
    torch.cuda.synchronize()
    q, g, k, v = st.parts(st.rows[0, L:L + 1])
    qn, _ = oracle.attn_norm_rope(q[0], k[0], st.qn, st.kn, L, NH, NKV, HD, ROT, 1.0e7)
    kc, vc = host(cache[0][0, :L + 1]), host(cache[1][0, :L + 1])
    if int8:
        kc = kc * host(cache[2][0, :L + 1])[..., None]
        vc = vc * host(cache[3][0, :L + 1])[..., None]
    ref = oracle.attn_token(qn, g[0], kc, vc, NH, NKV, HD)
    # INT8 cache: f16 MFMA operands for q and p (2^-11); FP32 cache: FP32 throughout
    assert relerr(host(out)[0], ref) <= (5e-3 if int8 else 2e-5)


def test_attn_position_outside_cache_flags(qw, ctx, oracle):
    """A token past the capacity writes nothing, outputs zeros and sets the
    device error flag; the other sequence in the launch is unaffected."""
    st = Stream(oracle, 2, 1, 500)
    cache = qw.kv_cache(2, 8, int8=True)
    ctx.device_error()  # clear
    out = run_gpu(qw, ctx, st, cache, dev(st.rows[:, 0]), [0, 8], 1, 1.0e7, ROT)
    torch.cuda.synchronize()
    assert ctx.device_error() != 0
    assert not host(out)[1].any() and host(out)[0].any()
    assert not host(cache[0][1]).any()



def test_attn_repeatable(qw, ctx, oracle):
    st = Stream(oracle, 2, 20, 600)
    outs = []
    for _ in range(3):
        cache = qw.kv_cache(2, 32, int8=True)
        outs.append(run_gpu(qw, ctx, st, cache, dev(st.rows.reshape(40, -1)), [0, 0], 20, 1.0e7, ROT))
    torch.cuda.synchronize()
    assert all(torch.equal(outs[0], o) for o in outs[1:])


def test_attn_errors(qw, ctx, oracle):
    st = Stream(oracle, 1, 1, 700)
    cache = qw.kv_cache(1, 8, int8=False)
    with pytest.raises(qw.QwError):  # 5 query heads per KV head
        run_gpu(qw, ctx, Stream(oracle, 1, 1, 701, nh=10), cache, dev(Stream(oracle, 1, 1, 701, nh=10).rows[:, 0]),
                [0], 1, 1.0e7, ROT)
    with pytest.raises(qw.QwError):  # odd rotary dim
        run_gpu(qw, ctx, st, cache, dev(st.rows[:, 0]), [0], 1, 1.0e7, 63)


def _ctx_with(qw, env, **kw):
    import os
    os.environ.update(env)
    try:
        return qw.Context(0, **kw)
    finally:
        for k in env:
            del os.environ[k]


@pytest.mark.parametrize("int8", [True, False])
def test_attn_prefill_kernel_matches_split_path(qw, oracle, relerr, int8):
    """The query-block prefill kernel, the key-split kernel (a context that
    sends every run to it) and, with a 6 MB workspace, the prefill kernel in
    768-token chunks of one sequence give the same result: 2 sequences of
    1000 tokens, the second starting at position 7 after a 7-token prefix.
    Over an INT8 cache the prefill kernel runs f16 MFMAs (q and p rounded to
    f16, 2^-11), so it meets the split path within the INT8 bar (5e-3); over
    an FP32 cache both are FP32 (2e-5); the chunked run is the same kernel."""
    B, T, cap = 2, 1000, 1024
    st = Stream(oracle, B, T + 7, 800)
    outs = []
    ctxs = [_ctx_with(qw, {}), _ctx_with(qw, {"QW_ATTN_PREFILL_MIN": "100000"}),
            _ctx_with(qw, {}, workspace_bytes=qw.lib().qw_workspace_query(1, 1, 1) + (6 << 20))]
    for c in ctxs:
        cache = qw.kv_cache(B, cap, int8=int8)
        sub = tuple(x[1:2] for x in cache)
        run_gpu(qw, c, st, sub, dev(st.rows[1, :7]), [0], 7, 1.0e7, ROT)
        rows = np.stack([st.rows[0, :T], st.rows[1, 7:T + 7]]).reshape(B * T, -1)
        outs.append(host(run_gpu(qw, c, st, cache, dev(rows), [0, 7], T, 1.0e7, ROT)))
        torch.cuda.synchronize()
    for c in ctxs:
        c.close()
    print("prefill vs split", int8, relerr(outs[1], outs[0]), relerr(outs[2], outs[0]))
    assert relerr(outs[1], outs[0]) <= (5e-3 if int8 else 2e-5) and relerr(outs[2], outs[0]) <= 2e-5
    ref0, _ = oracle_stream(oracle, st, st.rows[0, :200], int8, 1.0e7, ROT, cap)
    assert relerr(outs[0][:200], ref0) <= (5e-3 if int8 else 2e-5)


@pytest.mark.parametrize("io", ["f32", "bf16"])
def test_attn_one_launch_decode_matches_three_launches(qw, oracle, io):
    """One new token per sequence over an INT8 cache runs as one launch (the
    attention kernel normalizes q, writes the new K/V and merges its splits
    itself).  It computes exactly what the prep / split / combine launches
    compute: the same outputs and the same cache contents, bit for bit, over
    a prefill and 6 decode steps of 3 sequences at ragged positions -- short
    rows (one split) and long rows (9 splits) in the same launches."""
    B, cap = 3, 1200
    starts = [5, 300, 1100]
    st = Stream(oracle, B, max(starts) + 6, 900)
    tdt = torch.float32 if io == "f32" else torch.bfloat16
    res = []
    for env in ({}, {"QW_ATTN_FUSED": "0"}):
        c = _ctx_with(qw, env)
        cache = qw.kv_cache(B, cap, int8=True)
        for b in range(B):  # prefill each sequence's prefix (same kernels for both contexts)
            sub = tuple(x[b:b + 1] for x in cache)
            run_gpu(qw, c, st, sub, dev(st.rows[b, :starts[b]], tdt), [0], starts[b], 1.0e7, ROT)
        outs = []
        for s in range(6):
            rows = np.stack([st.rows[b, starts[b] + s] for b in range(B)])
            outs.append(run_gpu(qw, c, st, cache, dev(rows, tdt), [p + s for p in starts], 1, 1.0e7, ROT,
                                out_dtype=tdt))
        torch.cuda.synchronize()
        assert c.device_error() == 0
        res.append(([o.clone() for o in outs], [x.clone() for x in cache]))
        c.close()
    (o1, c1), (o0, c0) = res
    for s in range(6):
        assert torch.equal(o1[s], o0[s]), s
    for x1, x0 in zip(c1, c0):
        assert torch.equal(x1, x0)


@pytest.mark.parametrize("hd,nh,nkv,B,T,starts,io,vmul", [
    (256, 8, 2, 1, 32, [0], "f32", 1.0),          # the shortest run that takes it
    (256, 8, 2, 1, 65, [700], "f32", 1.0),        # a one-token block behind a prefix, masked tiles in several shares
    (256, 8, 2, 2, 300, [5, 600], "bf16", 1.0),   # ragged starts, blocks of several shares
    (256, 8, 2, 5, 40, [0, 1, 31, 32, 33], "f16", 1.0),  # more sequences than blocks
    (256, 8, 2, 70, 100, None, "f32", 1.0),       # more blocks than CUs: uncut blocks write the output themselves
    (256, 6, 2, 1, 130, [17], "f32", 1.0),        # three query heads per KV head
    (256, 2, 2, 2, 64, [0, 63], "f32", 1.0),      # one
    (128, 8, 2, 2, 200, [0, 90], "f32", 1.0),
    (256, 8, 2, 1, 150, [40], "f32", 1.0e6),      # V scales past the raise threshold's range
    (256, 8, 2, 3, 64, [0, 900, 1000], "f32", 1.0),  # one sequence runs past the capacity
])
def test_attn_prefill_blocks(qw, oracle, relerr, hd, nh, nkv, B, T, starts, io, vmul):
    """The 64-token-block INT8 prefill (expanded cache, shares, merge) against
    the 16-token kernels (a context that keeps every run on them; those are
    checked against the oracle above), over a cache with random codes behind the
    starts: edges of blocks and tiles, head groups, unaligned rows (odd column
    offset), the device error flag.  Both round q and p to f16 (2^-11) and sum
    in FP32, p against different maxima: 1e-3 normwise of each other; the cache
    written is the same kernel's and equal bit for bit."""
    cap = 1024 if T < 1000 else T
    starts = starts or [(37 * b) % 500 for b in range(B)]
    st = Stream(oracle, B, T, 900 + T + hd, hd=hd, nh=nh, nkv=nkv)
    tdt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[io]
    rows = dev(st.rows.reshape(B * T, -1))
    rows[:, nh * 2 * hd + nkv * hd:] *= vmul
    for pad in (0, 1):
        wide = torch.zeros(B * T, st.ld + 4, device="cuda", dtype=tdt)
        wide[:, pad:pad + st.ld] = rows.to(tdt)
        gen = torch.Generator(device="cuda").manual_seed(3)
        first = qw.kv_cache(B, cap, nkv, hd)
        for c in first[:2]:
            c.copy_(torch.randint(-127, 128, c.shape, generator=gen, device="cuda", dtype=torch.int8))
        for c, m in zip(first[2:], (1.0, vmul)):
            c.copy_(torch.rand(c.shape, generator=gen, device="cuda") * 0.02 * m + 0.001)
        outs, caches, flags = [], [], []
        for env in ({"QW_ATTN_PF_MIN": "32"}, {"QW_ATTN_PF_MIN": "1000000"}):
            c = _ctx_with(qw, env)
            cache = tuple(x.clone() for x in first)
            outs.append(run_gpu(qw, c, st, cache, wide[:, pad:], starts, T, 1.0e7, hd // 4,
                                out_dtype=torch.float32 if vmul > 1 else tdt, max_len=cap))
            flags.append(c.device_error())
            torch.cuda.synchronize()
            caches.append(cache)
            c.close()
        assert flags[0] == flags[1] and (flags[0] != 0) == any(s + T > cap for s in starts)
        assert all(torch.equal(x, y) for x, y in zip(*caches))
        err = relerr(host(outs[0]), host(outs[1]))
        print("blocks", hd, nh, nkv, B, T, pad, err)
        assert err <= (1e-3 if io == "f32" else 8e-3 if io == "bf16" else 2e-3), err


def _random_cache(qw, B, cap, seed=3):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    cache = qw.kv_cache(B, cap)
    for c in cache[:2]:
        c.copy_(torch.randint(-127, 128, c.shape, generator=gen, device="cuda", dtype=torch.int8))
    for c in cache[2:]:
        c.copy_(torch.rand(c.shape, generator=gen, device="cuda") * 0.02 + 0.001)
    return cache


@pytest.mark.parametrize("B,T,cap,start,mb", [
    (1, 64, 16384, 16250, 0),  # a block cut into 85 shares: the newest keys are its last one
    (1, 128, 8192, 8000, 0),
    (1, 192, 32768, 5280, 0),  # a cache much longer than the contexts
    (4, 64, 4096, 3968, 0),
    (1, 64, 32768, 0, 0),
    # workspaces (MiB) that cut the call: a plan for 4 CUs, one sequence at a time;
    # 2 sequences, then 1; 96 tokens of a sequence at a time; every unit a partial; a
    # plan for 86 CUs
    (3, 200, 1024, 700, 5), (3, 200, 1024, 800, 8), (3, 200, 1024, 824, 10), (3, 200, 1024, 0, 12),
    (3, 200, 1024, 500, 32),
])
def test_attn_prefill_blocks_plan(qw, oracle, relerr, B, T, cap, start, mb):
    """Contexts where the plan of the 64-token blocks is tight (shares just below
    the units its grid has room for) and workspaces that cut the call into
    segments, against the 16-token kernels and, the last query of each sequence,
    against the oracle's attention over the cache as written.  A first call over
    NaN scales fills the workspace's partials, so that a share nobody computed
    shows."""
    st = Stream(oracle, B, T, 3100 + T)
    rows = dev(st.rows.reshape(B * T, -1))
    first = _random_cache(qw, B, cap)
    kw = {"workspace_bytes": qw.lib().qw_workspace_query(1, 1, 1) + (mb << 20)} if mb else {}
    outs = []
    for env in ({"QW_ATTN_PF_MIN": "32"}, {"QW_ATTN_PF_MIN": "1000000"}):
        c = _ctx_with(qw, env, **kw)
        cache = tuple(x.clone() for x in first)
        nan = (cache[0], cache[1], torch.full_like(cache[2], float("nan")), torch.full_like(cache[3], float("nan")))
        run_gpu(qw, c, st, nan, rows, [start] * B, T, 1.0e7, ROT, max_len=cap)
        cache = tuple(x.clone() for x in first)
        outs.append(host(run_gpu(qw, c, st, cache, rows, [start] * B, T, 1.0e7, ROT, max_len=cap)))
        assert c.device_error() == 0
        c.close()
    err = relerr(outs[0], outs[1])
    print("plan", B, T, cap, start, mb, err)
    assert err <= 1e-3, err  # as test_attn_prefill_blocks
    P = start + T - 1
    for b in range(B):
        q, g, k, _ = st.parts(st.rows[b, T - 1:T])
        qn, _ = oracle.attn_norm_rope(q[0], k[0], st.qn, st.kn, P, NH, NKV, HD, ROT, 1.0e7)
        kc, vc = (host(cache[i][b, :P + 1]) * host(cache[i + 2][b, :P + 1])[..., None] for i in (0, 1))
        ref = oracle.attn_token(qn, g[0], kc, vc, NH, NKV, HD)
        assert relerr(outs[0].reshape(B, T, -1)[b, -1], ref) <= 5e-3, b


@pytest.mark.parametrize("B,T,cap,starts,hd,io", [
    (1, 16, 600, [500], 256, "f32"),           # one block, its keys cut
    (1, 300, 1024, [700], 256, "f32"),         # up to the last cache slot
    (2, 90, 700, [0, 600], 256, "bf16"),       # one share and several in one launch, ragged blocks
    (1, 200, 900, [650], 128, "f32"),
    (2, 64, 640, [100, 600], 256, "f32"),      # the second sequence runs past the capacity
])
def test_attn_prefill_f32_shares(qw, oracle, relerr, B, T, cap, starts, hd, io):
    """The FP32 query-block kernel with its keys cut into shares against the
    key-split row kernel (a context that sends every run to it), over a random
    cache; rows with an odd column offset take the element accesses.  FP32
    throughout: 2e-5 normwise (BF16 outputs: one rounding)."""
    st = Stream(oracle, B, T, 1700 + T, hd=hd)
    tdt = {"f32": torch.float32, "bf16": torch.bfloat16}[io]
    for pad in (0, 1):
        wide = torch.zeros(B * T, st.ld + 4, device="cuda", dtype=tdt)
        wide[:, pad:pad + st.ld] = dev(st.rows.reshape(B * T, -1)).to(tdt)
        gen = torch.Generator(device="cuda").manual_seed(5)
        first = [torch.randn(B, cap, 2, hd, generator=gen, device="cuda") for _ in range(2)]
        outs, caches, flags = [], [], []
        for env in ({}, {"QW_ATTN_PREFILL_MIN": "100000"}):
            c = _ctx_with(qw, env)
            zero = torch.zeros(B, cap, 2, device="cuda")
            cache = (first[0].clone(), first[1].clone(), zero, zero)
            outs.append(run_gpu(qw, c, st, cache, wide[:, pad:], starts, T, 1.0e7, hd // 4, out_dtype=tdt, max_len=cap))
            flags.append(c.device_error())
            torch.cuda.synchronize()
            caches.append(cache)
            c.close()
        assert flags[0] == flags[1] and (flags[0] != 0) == any(s + T > cap for s in starts)
        assert torch.equal(caches[0][0], caches[1][0]) and torch.equal(caches[0][1], caches[1][1])
        err = relerr(host(outs[0]), host(outs[1]))
        print("f32 shares", B, T, cap, hd, pad, err)
        assert err <= (2e-5 if io == "f32" else 8e-3), err


@pytest.mark.parametrize("int8,hd,io", [(True, 256, "f32"), (True, 256, "bf16"), (True, 256, "f16"), (True, 128, "f32"),
                                        (False, 256, "bf16")])
def test_attn_prefill_lone_split_rows(qw, ctx, oracle, relerr, int8, hd, io):
    """16-token blocks whose keys are one split write the output themselves, four
    dims per access or, for rows at an odd column, by elements: the same values
    (1e-6, the same FP32 steps; 16-bit outputs equal), and the oracle's."""
    B, T, cap = 2, 61, 64
    st = Stream(oracle, B, T, 2500 + hd, hd=hd)
    tdt = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}[io]
    rows = dev(st.rows.reshape(B * T, -1)).to(tdt)
    outs = []
    for pad in (0, 1):
        wide = torch.zeros(B * T, st.ld + 4, device="cuda", dtype=tdt)
        wide[:, pad:pad + st.ld] = rows
        cache = qw.kv_cache(B, cap, st.nkv, hd, int8=int8)
        outs.append(host(run_gpu(qw, ctx, st, cache, wide[:, pad:], [0, 3], T, 1.0e7, hd // 4, out_dtype=tdt)))
    assert relerr(outs[0], outs[1]) <= (1e-6 if io == "f32" else 0.0)
    ref, _ = oracle_stream(oracle, st, host(rows).reshape(B, T, -1)[0], int8, 1.0e7, hd // 4, cap)
    assert relerr(outs[0].reshape(B, T, -1)[0], ref) <= (5e-3 if io == "f32" else 1e-2)


@pytest.mark.parametrize("B,T", [(1, 16), (2, 40), (2, 150)])
def test_attn_prefill_f32_smallest_workspace(qw, oracle, relerr, B, T):
    """24 heads of 256 over an FP32 cache in the smallest workspace (3 MB): one row
    of normalized q is 24 KB, with 8 key shares' partials 218 KB.  16 tokens fit
    only with fewer shares, 2 x 40 with one, 2 x 150 with one and in segments of 128
    tokens; against the default workspace (FP32 throughout, 2e-5)."""
    nh, nkv, cap, start = 24, 6, 1100, 930
    st = Stream(oracle, B, T, 2700 + T, nh=nh, nkv=nkv)
    gen = torch.Generator(device="cuda").manual_seed(7)
    first = [torch.randn(B, cap, nkv, HD, generator=gen, device="cuda") for _ in range(2)]
    outs = []
    for kw in ({}, {"workspace_bytes": 1}):
        c = _ctx_with(qw, {}, **kw)
        zero = torch.zeros(B, cap, nkv, device="cuda")
        cache = (first[0].clone(), first[1].clone(), zero, zero)
        outs.append(host(run_gpu(qw, c, st, cache, dev(st.rows.reshape(B * T, -1)), [start] * B, T, 1.0e7, ROT)))
        assert c.device_error() == 0
        c.close()
    assert relerr(outs[1], outs[0]) <= 2e-5


@pytest.mark.parametrize("int8,T,hd", [(False, 1, 256), (True, 1, 256), (True, 40, 256), (True, 20, 128), (True, 1, 128)])
def test_attn_key_norm_rounding(qw, oracle, int8, T, hd):
    """The keys' norm is summed in one order by every kernel that writes the
    cache (the row kernel, its four-row form, the one-launch decode): per lane
    x1^2, then x0^2, x2^2, x3^2 fused onto it, then lanes 32, 16, .. 1 apart.
    FP32 cache: the keys bit for bit; INT8: their scales.  The keys have 13
    fraction bits, so that squares and partial sums are exact in double and
    each step below rounds once."""
    B, nkv, E = 96 // min(T, 4), 2, hd // 64
    st = Stream(oracle, B, T, 2300 + hd, hd=hd)
    rows = np.round(st.rows * 8192.0).astype(np.float32) / np.float32(8192.0)
    c = _ctx_with(qw, {"QW_ATTN_PF_MIN": "32"})
    cache = qw.kv_cache(B, T, nkv, hd, int8=int8)
    run_gpu(qw, c, st, cache, dev(rows.reshape(B * T, -1)), [0] * B, T, 1.0e7, 0)
    torch.cuda.synchronize()
    c.close()
    f32, f64 = np.float32, np.float64
    k = rows[..., st.nh * 2 * hd:st.nh * 2 * hd + nkv * hd].reshape(B, T, nkv, hd)
    x = k.reshape(B, T, nkv, 64, E)
    sq = x.astype(f64) ** 2
    ss = (sq[..., 0] + sq[..., 1].astype(f32)).astype(f32)
    for e in range(2, E):
        ss = (sq[..., e] + ss).astype(f32)
    lane = np.arange(64)
    for off in (32, 16, 8, 4, 2, 1):
        ss = ss + ss[..., lane ^ off]
    rms = np.sqrt(((ss[..., :1] / f32(hd)).astype(f64) + f64(f32(1e-6))).astype(f32))
    y = k / rms * (f32(1.0) + st.kn)
    if int8:
        m = np.abs(y).max(axis=-1) / f32(127.0)
        assert np.array_equal(host(cache[2]), m)
    else:
        assert np.array_equal(host(cache[0]), y)
