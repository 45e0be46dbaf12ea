"""GPU parity of the direct-A GEMM over INT8 weights and F16 activations
(qw_gemm_da.hip: units converted to f16 in registers, row scales on the
accumulators) in its 4-wave, 8-wave and split-K forms, against FP64 on the
stored codes, scales and F16 activations and against the LDS-staged INT8 GEMM
(QW_GEMM_DA=0), plus bit-identical repeats.

The GLU rows' split runs where their blocks are fewer than half the CUs (1040 rows
of 520 here); 3584 make half a block per CU and more and are never split.

Sizes: ragged token blocks (1, 127, 129 past a block), ragged row blocks
(1008 = 63 tiles, 520), K = 1024 / 2048 / 3584 (8..28 rounds of the two-unit
ring) and K = 128 (one round).  Bars: codes are exact in f16, products of f16
pairs exact in FP32, so the error is that of K FP32 additions in MFMA order: 2e-5
normwise vs FP64, 1e-5 vs the other route; 1e-4 through SiLU.
"""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(a, dtype=torch.float32):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").to(dtype)


def host(t):
    return t.float().cpu().numpy()


FORMS = {"off": {"QW_GEMM_DA": "0"},
         "w4": {"QW_GEMM_DA": "2", "QW_GEMM_DA_W8": "0"},
         "w8": {"QW_GEMM_DA": "2", "QW_GEMM_DA_W8": "1"},
         "s2": {"QW_GEMM_DA_SPLIT": "2"}, "s7": {"QW_GEMM_DA_SPLIT": "7"}, "s8": {"QW_GEMM_DA_SPLIT": "8"}}


@pytest.fixture(scope="module")
def ctx_f(qw):
    made = {}

    def get(form):
        if form not in made:
            env = dict(FORMS[form], QW_GEMM_MIN_M="33", QW_GEMM_ROWS="256")
            old = {k: os.environ.get(k) for k in env}
            os.environ.update(env)
            try:
                made[form] = qw.Context(0)
            finally:
                for k, v in old.items():
                    os.environ.pop(k, None) if v is None else os.environ.__setitem__(k, v)
        return made[form]
    yield get
    for c in made.values():
        c.close()


def codes(oracle, W):
    q, s = oracle.quantize_rowscale(W)
    return q.astype(np.float64) * s.astype(np.float64)[:, None]


@pytest.mark.parametrize("N,K,M,form", [
    (1024, 3584, 1000, "w4"), (1024, 3584, 1000, "w8"), (1024, 3584, 1000, "s7"), (1024, 3584, 520, "s2"),
    (1024, 2048, 777, "s8"), (1008, 1024, 129, "w4"), (520, 1024, 255, "w8"), (1008, 128, 40, "w4"),
    (6160, 1024, 257, "w8"), (520, 1024, 300, "s2")])
def test_i8_direct_a_residual(qw, ctx_f, oracle, relerr, N, K, M, form):
    W = oracle.normal((N, K), 8100 + K + N, 0.0, 0.02) * (1.0 + np.arange(N, dtype=np.float32)[:, None] / 64)
    x = oracle.normal((M, K), 8101 + M)
    r = oracle.normal((M, N), 8102)
    xt = dev(x, torch.float16)
    outs = []
    for f in (form, form, "off"):
        ctx = ctx_f(f)
        w = qw.Weight.pack(ctx, W, qw.WFMT_INT8)
        y = dev(r)
        qw.linear(ctx, w, xt, y, residual=y)
        torch.cuda.synchronize()
        assert ctx.device_error() == 0
        outs.append(y)
    assert torch.equal(outs[0], outs[1]), "repeat differs"
    prod = host(xt).astype(np.float64) @ codes(oracle, W).T
    assert relerr(host(outs[0]), prod + r) <= 2e-5
    assert relerr(host(outs[0]), host(outs[2]).astype(np.float64)) <= 1e-5


@pytest.mark.parametrize("N,M", [(6160, 2500), (4096, 4096), (4096, 900)])
def test_i8_route_by_rounds(qw, ctx, oracle, relerr, N, M):
    """The unforced route where the 8-wave blocks' last round is nearly empty (260
    blocks), where it is full (256), and at exactly half a block per CU, against FP64."""
    K = 128
    W = oracle.normal((N, K), 8150 + N, 0.0, 0.02)
    xt = dev(oracle.normal((M, K), 8151 + M), torch.float16)
    w = qw.Weight.pack(ctx, W, qw.WFMT_INT8)
    y = torch.empty(M, N, device="cuda")
    qw.linear(ctx, w, xt, y)
    torch.cuda.synchronize()
    assert ctx.device_error() == 0
    assert relerr(host(y), host(xt).astype(np.float64) @ codes(oracle, W).T) <= 2e-5


@pytest.mark.parametrize("I,M,form", [(3584, 600, "w4"), (3584, 513, "w8"), (520, 200, "w4"), (3584, 520, "s2"), (520, 200, "s2"),
                                      (520, 129, "s2")])
def test_i8_direct_a_glu(qw, ctx_f, oracle, relerr, I, M, form):
    H = 1024
    G = oracle.normal((I, H), 8130, 0.0, 0.02)
    U = oracle.normal((I, H), 8131, 0.0, 0.02)
    xt = dev(oracle.normal((M, H), 8133 + M), torch.float16)
    def run(form):
        ctx = ctx_f(form)
        w = qw.Weight.pack_glu(ctx, G, U, qw.WFMT_INT8)
        h = torch.empty(M, I, device="cuda")
        qw.linear(ctx, w, xt, h)
        torch.cuda.synchronize()
        assert ctx.device_error() == 0
        return h
    h = run(form)
    if form == "s2":  # two sums of half the terms round otherwise than one: whether the split ran
        assert torch.equal(h, run("w4")) == (I == 3584)
    xs = host(xt).astype(np.float64)
    g, u = xs @ codes(oracle, G).T, xs @ codes(oracle, U).T
    assert relerr(host(h), g / (1.0 + np.exp(-g)) * u) <= 1e-4
