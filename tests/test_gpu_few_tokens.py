"""The few-token path (csrc/qlinear_sm.h): at most 128 tokens, or 1024 while the products are small, the
layer's forward and backward run as two launches each, the products' reductions dealt over ranges.

At the edges of its tiles (32, 64, 128 tokens) and ranges, over the weight forms, ranks, output types and
an unaligned output, it is held to the path for more tokens (R97Q_DECODE_FUSED asks for it): the decoded
weights are the same bf16 values and every product is exact in f32, so the two differ by the order of f32
sums of K or N terms and by the [hi | lo] bf16 split (16 bits) of the adapter's activations there --
2e-5 relative, and a bf16 output by its own rounding (2^-8). Values against the float64 host rows are
tests/test_gpu_qlinear.py's (its cases run this path too)."""
import ctypes as C

import numpy as np
import pytest
import torch

import iqr_synth as S
from gpu_util import bf16_tensor, device_desc, prepared

pytestmark = pytest.mark.gpu


@pytest.fixture
def modes():
    from r9700training_amd import R97Q_DECODE_AUTO, R97Q_DECODE_FUSED, lib

    L = lib()
    yield lambda few: L.r97q_set_decode_once(R97Q_DECODE_AUTO if few else R97Q_DECODE_FUSED)
    assert L.r97q_set_decode_once(R97Q_DECODE_AUTO) >= 0


def _weight(N, K, bits, run, codes8, seed, keep):
    from r9700training_amd.qlinear import QWeight

    rng = np.random.default_rng(seed)
    p = S.trellis(rows=N, cols=K, bits=bits, run_rows=run, rowf=True, seed=seed, packed=True,
                  scale_col=(0.75 + 0.5 * rng.random(K // 128)).astype(np.float32))
    if not codes8:
        return prepared(p, keep)
    sc = torch.from_numpy(p.scale_col).cuda()
    keep.append(sc)
    return QWeight(device_desc(p, keep), scale_col=sc, codes8=True)


def _rel(a, b):
    return float((a.double() - b.double()).norm() / b.double().norm())


CASES = [
    # T, N, K, r, bits, run, codes8, bf16 out
    (1, 128, 128, 0, 5, 128, False, False),     # one range of two steps
    (1, 384, 2048, 16, 5, 256, False, True),    # a short last run, many ranges
    (31, 512, 640, 8, 3, 64, False, False),
    (32, 640, 512, 64, 4, 96, False, False),
    (33, 256, 384, 32, 6, 32, False, True),
    (64, 1024, 256, 16, 5, 256, True, False),
    (65, 128, 1152, 64, 6, 128, False, False),
    (128, 384, 384, 8, 4, 256, False, False),
    (129, 512, 768, 16, 5, 256, False, True),   # past the unconditional line, two token tiles
    (500, 640, 896, 64, 5, 128, True, False),
    (512, 2048, 2048, 16, 5, 256, False, False),  # 8 steps a CU, and 32 for each below
    (512, 4096, 4096, 32, 5, 256, False, False),
    (1000, 2048, 4096, 8, 4, 256, True, True),
    (1024, 256, 512, 32, 3, 256, False, False),  # the most tokens
    (700, 6144, 128, 64, 5, 256, False, False),  # the forward past its line, the backward within
    (846, 256, 6144, 8, 4, 128, True, False),    # and the other way round
]


@pytest.mark.parametrize("T,N,K,r,bits,run,codes8,bf16", CASES)
def test_few_tokens_match_the_other_path(modes, T, N, K, r, bits, run, codes8, bf16):
    from r9700training_amd.qlinear import qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case few tokens T={T} N={N} K={K} r={r} bits={bits} codes8={codes8} bf16={bf16}", flush=True)
    rng = np.random.default_rng(T + N + K)
    keep = []
    w = _weight(N, K, bits, run, codes8, T + bits, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A = bf16_tensor(0.01 * rng.standard_normal((r, K))) if r else None
    B = bf16_tensor(0.01 * rng.standard_normal((N, r))) if r else None
    dt = torch.bfloat16 if bf16 else torch.float32
    base = torch.randn((T, K), device="cuda").to(dt)
    got = {}
    for few in (True, False):
        modes(few)
        # outputs one element past an aligned start take the value-by-value stores
        y = torch.empty(T * N + 1, dtype=dt, device="cuda")[few:][: T * N].view(T, N)
        dx = torch.empty(T * K + 1, dtype=dt, device="cuda")[few:][: T * K].view(T, K).copy_(base)
        Y, t = qlinear_lora_fwd(w, X, A, B, 2.0, out=y)
        Y2, _ = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=dt)
        assert torch.equal(Y, Y2)
        dA = torch.ones((r, K), device="cuda") if r else None
        dB = torch.ones((N, r), device="cuda") if r else None
        dX, dA, dB = qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dX=dx, accumulate=True, dA=dA, dB=dB)
        dX2, dA2, dB2 = qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dX=base.clone(), accumulate=True)
        assert torch.equal(dX, dX2)
        if r:
            assert torch.allclose(dA, dA2 + 1) and torch.allclose(dB, dB2 + 1)
        got[few] = (Y, dX) if not r else (Y, dX, t, dA2, dB2)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(got[True], got[False])):
        e = _rel(a, b)
        assert torch.isfinite(a).all() and e <= (2 ** -8 if bf16 and i < 2 else 2e-5), (i, e)


@pytest.mark.parametrize("N,K,r,most", [(1024, 1024, 8, 2048), (2048, 512, 64, 2048), (640, 896, 32, 4096),
                                        (256, 256, 0, 1536)])
@pytest.mark.parametrize("T", [1, 128, 777, 1024])
def test_workspace_of_a_larger_batch(modes, N, K, r, most, T):
    """One workspace sized for `most` tokens serves the smaller batches, which may ask for more than it:
    the bits are the few-token path's where its layout fits and the other path's where not, for the
    fused and the stage entries alike, and nothing past the stated bytes is written. Less than either
    path needs is still refused."""
    from r9700training_amd import R97Q_F32, R97qError, _ptr, _stream, check, lib
    from r9700training_amd.qlinear import qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case workspace of {most} tokens, T={T} N={N} K={K} r={r}", flush=True)
    rng = np.random.default_rng(T + N)
    keep = []
    w = _weight(N, K, 5, 128, False, T + N, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A = bf16_tensor(0.01 * rng.standard_normal((r, K))) if r else None
    B = bf16_tensor(0.01 * rng.standard_normal((N, r))) if r else None
    L, P, st = lib(), _ptr, _stream()
    kw = dict(dx_dtype=torch.float32)
    modes(False)
    need = [f(T, N, K, r) for f in (L.r97q_fwd_workspace_bytes, L.r97q_bwd_workspace_bytes)]
    Yo, to = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.float32)
    other = (Yo, *qlinear_lora_bwd(w, X, dY, A, B, to, 2.0, **kw))
    modes(True)
    Yf, tf = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.float32)
    own = (Yf, *qlinear_lora_bwd(w, X, dY, A, B, to, 2.0, **kw))
    asked = [f(T, N, K, r) for f in (L.r97q_fwd_workspace_bytes, L.r97q_bwd_workspace_bytes)]
    held = [f(most, N, K, r) for f in (L.r97q_fwd_workspace_bytes, L.r97q_bwd_workspace_bytes)]
    buf = [torch.full((max(h, n) + 4096,), 0xA5, dtype=torch.uint8, device="cuda") for h, n in zip(held, need)]
    ws = [b[:h] for b, h in zip(buf, held)]
    Y, t = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.float32, workspace=ws[0])
    got = (Y, *qlinear_lora_bwd(w, X, dY, A, B, to, 2.0, workspace=ws[1], **kw))
    Ys, dXs = torch.empty_like(Y), torch.empty_like(got[1])
    ts = torch.empty_like(t) if r else None
    dAs, dBs = (torch.zeros_like(got[2]), torch.zeros_like(got[3])) if r else (None, None)
    f, b = (P(ws[0]), held[0], st), (P(ws[1]), held[1], st)
    check(L.r97q_lora_fwd_prep(T, N, K, P(X), P(A), r, 2.0, P(ts), *f), "fwd_prep")
    check(L.r97q_qlinear_fwd_base(C.byref(w.w), P(X), T, P(B), r, P(Ys), R97Q_F32, *f), "fwd_base")
    check(L.r97q_lora_bwd_prep(T, N, K, P(dY), P(A), P(B), P(to), r, 2.0, *b), "bwd_prep")
    check(L.r97q_lora_bwd_grads(T, N, K, P(X), P(dY), r, P(dAs), P(dBs), *b), "bwd_grads")
    check(L.r97q_qlinear_dx_base(C.byref(w.w), P(dY), T, r, P(dXs), R97Q_F32, 0, *b), "dx_base")
    torch.cuda.synchronize()
    for bb, h in zip(buf, held):
        assert (bb[h:] == 0xA5).all()
    staged = (Ys, dXs, dAs, dBs)
    for i in range(4 if r else 2):
        one = 0 if i == 0 else 1
        assert torch.equal(got[i], own[i]) or torch.equal(got[i], other[i]), i
        assert torch.equal(staged[i], own[i]) or torch.equal(staged[i], other[i]), i
        if held[one] >= asked[one]:
            assert torch.equal(got[i], own[i]) and torch.equal(staged[i], own[i]), i
    for one, short in enumerate(min(n, a) for n, a in zip(need, asked)):
        with pytest.raises(R97qError):
            # the fused entries need no more than the stages' part past the partials
            small = buf[one][: short // 8]
            if one == 0:
                qlinear_lora_fwd(w, X, A, B, 2.0, workspace=small)
            else:
                qlinear_lora_bwd(w, X, dY, A, B, to, 2.0, workspace=small)


@pytest.mark.parametrize("over", ["X", "dY"])
@pytest.mark.parametrize("T,r", [(5, 8), (130, 16), (300, 64)])
def test_outputs_over_their_inputs(T, r, over):
    """A bf16 Y written over X and a bf16 dX over X or dY (a square layer): the separate buffers' bits,
    the factor gradients included, as on the path for more tokens."""
    from r9700training_amd.qlinear import qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case few tokens in place T={T} r={r} over={over}", flush=True)
    rng = np.random.default_rng(T)
    keep = []
    N = K = 512
    w = _weight(N, K, 5, 128, False, T, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A, B = bf16_tensor(0.01 * rng.standard_normal((r, K))), bf16_tensor(0.01 * rng.standard_normal((N, r)))
    Y, t = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.bfloat16)
    want = (Y, *qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dx_dtype=torch.bfloat16))
    y = X.clone()
    qlinear_lora_fwd(w, y, A, B, 2.0, out=y)
    x, g = X.clone(), dY.clone()
    dX, dA, dB = qlinear_lora_bwd(w, x, g, A, B, t, 2.0, dX=x if over == "X" else g)
    torch.cuda.synchronize()
    for a, b in zip((y, dX, dA, dB), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,r", [(5, 8), (130, 16), (300, 64)])
def test_dx_over_t(T, r):
    """An f32 dX whose buffer holds t: the separate buffers' bits, as on the path for more tokens."""
    from r9700training_amd.qlinear import qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case few tokens dX over t T={T} r={r}", flush=True)
    rng = np.random.default_rng(T)
    keep = []
    N, K = 512, 384
    w = _weight(N, K, 5, 128, False, T, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A, B = bf16_tensor(0.01 * rng.standard_normal((r, K))), bf16_tensor(0.01 * rng.standard_normal((N, r)))
    _, t = qlinear_lora_fwd(w, X, A, B, 2.0)
    want = qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dx_dtype=torch.float32)
    dX = torch.empty_like(want[0])
    t2 = dX.view(-1)[: T * r].view(T, r).copy_(t)
    got = qlinear_lora_bwd(w, X, dY, A, B, t2, 2.0, dX=dX)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("T,N,K,r", [(7, 384, 512, 16), (130, 256, 384, 0), (300, 512, 256, 64)])
def test_stages_keep_their_operands(T, N, K, r):
    """The stage entries on this path: the fused entries' bits, with X and dY overwritten between the
    preparation and the product (the preparation holds them, as it holds the tiled copy on the path
    for more tokens), and the forward that allocates nothing the same bits."""
    from r9700training_amd import R97Q_F32, _ptr, _stream, check, lib
    from r9700training_amd.qlinear import bwd_workspace, fwd_workspace, qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case few tokens stages T={T} N={N} K={K} r={r}", flush=True)
    rng = np.random.default_rng(T)
    keep = []
    w = _weight(N, K, 5, 128, False, T, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A = bf16_tensor(0.01 * rng.standard_normal((r, K))) if r else None
    B = bf16_tensor(0.01 * rng.standard_normal((N, r))) if r else None
    Y, t = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.float32)
    dX, dA, dB = qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dx_dtype=torch.float32)
    L, P, st = lib(), _ptr, _stream()
    ws, wb = fwd_workspace(T, N, K, r), bwd_workspace(T, N, K, r)
    Ys, dXs = torch.empty_like(Y), torch.empty_like(dX)
    ts = torch.empty_like(t) if r else None
    x, g = X.clone(), dY.clone()
    check(L.r97q_lora_fwd_prep(T, N, K, P(x), P(A), r, 2.0, P(ts), P(ws), ws.numel(), st), "fwd_prep")
    x.fill_(float("nan"))
    check(L.r97q_qlinear_fwd_base(C.byref(w.w), P(x), T, P(B), r, P(Ys), R97Q_F32, P(ws), ws.numel(), st), "fwd_base")
    check(L.r97q_lora_bwd_prep(T, N, K, P(g), P(A), P(B), P(t), r, 2.0, P(wb), wb.numel(), st), "bwd_prep")
    dAs = torch.zeros_like(dA) if r else None
    dBs = torch.zeros_like(dB) if r else None
    check(L.r97q_lora_bwd_grads(T, N, K, P(X), P(g), r, P(dAs), P(dBs), P(wb), wb.numel(), st), "bwd_grads")
    g.fill_(float("nan"))
    check(L.r97q_qlinear_dx_base(C.byref(w.w), P(g), T, r, P(dXs), R97Q_F32, 0, P(wb), wb.numel(), st), "dx_base")
    Yn = torch.empty_like(Y)
    tn = torch.empty_like(t) if r else None
    check(L.r97q_qlinear_lora_fwd_noalloc(C.byref(w.w), P(X), T, P(A), P(B), r, 2.0, P(Yn), R97Q_F32, P(tn), st), "noalloc")
    torch.cuda.synchronize()
    assert torch.equal(Y, Ys) and torch.equal(dX, dXs) and torch.equal(Y, Yn)
    if r:
        assert torch.equal(t, ts) and torch.equal(dA, dAs) and torch.equal(dB, dBs) and torch.equal(t, tn)


@pytest.mark.parametrize("T", [40, 1100])
def test_backward_without_gradients(T):
    """Both factor gradients skipped (NULL) with an adapter: dX is the bits it is with them, on either path,
    from the fused and the stage entries."""
    from r9700training_amd import R97Q_F32, _ptr, _stream, check, lib
    from r9700training_amd.qlinear import bwd_workspace, qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case backward without gradients T={T}", flush=True)
    rng = np.random.default_rng(T)
    keep = []
    N, K, r = 256, 384, 16
    w = _weight(N, K, 5, 128, False, T, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A, B = bf16_tensor(0.01 * rng.standard_normal((r, K))), bf16_tensor(0.01 * rng.standard_normal((N, r)))
    L, P, st = lib(), _ptr, _stream()
    _, t = qlinear_lora_fwd(w, X, A, B, 2.0)
    want = qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dx_dtype=torch.float32)[0]
    ws = bwd_workspace(T, N, K, r)
    b = (P(ws), ws.numel(), st)
    dX, dXs = torch.empty_like(want), torch.empty_like(want)
    check(L.r97q_qlinear_lora_bwd(C.byref(w.w), P(X), P(dY), T, P(A), P(B), r, 2.0, P(t), P(dX), R97Q_F32, 0, None, None, *b),
          "bwd")
    check(L.r97q_lora_bwd_prep(T, N, K, P(dY), P(A), P(B), P(t), r, 2.0, *b), "bwd_prep")
    check(L.r97q_lora_bwd_grads(T, N, K, P(X), P(dY), r, None, None, *b), "bwd_grads")
    check(L.r97q_qlinear_dx_base(C.byref(w.w), P(dY), T, r, P(dXs), R97Q_F32, 0, *b), "dx_base")
    torch.cuda.synchronize()
    assert torch.equal(dX, want) and torch.equal(dXs, want)


@pytest.mark.parametrize("T,N,K,r", [(1, 384, 512, 8), (33, 256, 640, 32), (130, 256, 384, 16), (300, 512, 256, 64)])
def test_factor_off_its_alignment(T, N, K, r):
    """A in a view one, two or four elements past an aligned start (off 16 bytes, the last on 8): the fused
    entries, the stages and the forward that allocates nothing read it a value or half a piece at a
    time, the aligned A's bits."""
    from r9700training_amd import R97Q_F32, _ptr, _stream, check, lib
    from r9700training_amd.qlinear import bwd_workspace, qlinear_lora_bwd, qlinear_lora_fwd

    print(f"case few tokens unaligned A T={T} N={N} K={K} r={r}", flush=True)
    rng = np.random.default_rng(T)
    keep = []
    w = _weight(N, K, 5, 128, False, T, keep)
    X, dY = bf16_tensor(rng.standard_normal((T, K))), bf16_tensor(rng.standard_normal((T, N)))
    A, B = bf16_tensor(0.01 * rng.standard_normal((r, K))), bf16_tensor(0.01 * rng.standard_normal((N, r)))
    L, P, st = lib(), _ptr, _stream()
    Y, t = qlinear_lora_fwd(w, X, A, B, 2.0, y_dtype=torch.float32)
    want = (Y, t, *qlinear_lora_bwd(w, X, dY, A, B, t, 2.0, dx_dtype=torch.float32))
    for at in (1, 2, 4):
        Au = torch.empty(r * K + 8, dtype=torch.bfloat16, device="cuda")[at:][: r * K].view(r, K).copy_(A)
        Y2, t2 = qlinear_lora_fwd(w, X, Au, B, 2.0, y_dtype=torch.float32)
        got = (Y2, t2, *qlinear_lora_bwd(w, X, dY, Au, B, t, 2.0, dx_dtype=torch.float32))
        Yn, tn = torch.empty_like(Y), torch.empty_like(t)
        check(L.r97q_qlinear_lora_fwd_noalloc(C.byref(w.w), P(X), T, P(Au), P(B), r, 2.0, P(Yn), R97Q_F32, P(tn), st),
              "noalloc")
        ws = bwd_workspace(T, N, K, r)
        b = (P(ws), ws.numel(), st)
        dX, dA, dB = torch.empty_like(want[2]), torch.zeros_like(want[3]), torch.zeros_like(want[4])
        check(L.r97q_lora_bwd_prep(T, N, K, P(dY), P(Au), P(B), P(t), r, 2.0, *b), "bwd_prep")
        check(L.r97q_lora_bwd_grads(T, N, K, P(X), P(dY), r, P(dA), P(dB), *b), "bwd_grads")
        check(L.r97q_qlinear_dx_base(C.byref(w.w), P(dY), T, r, P(dX), R97Q_F32, 0, *b), "dx_base")
        torch.cuda.synchronize()
        for i, (g, x) in enumerate(zip((*got, Yn, tn, dX, dA, dB), (*want, *want))):
            assert torch.equal(g, x), (at, i)


@pytest.mark.parametrize("T,C,r", [(1, 128, 8), (33, 640, 64), (256, 384, 64), (257, 384, 32), (512, 256, 16),
                                   (512, 128, 64), (513, 128, 64), (768, 256, 32), (769, 256, 32), (1024, 256, 16),
                                   (1025, 256, 8)])
@pytest.mark.parametrize("off", [False, True])
def test_adapter_adjoints(T, C, r, off):
    """The adapter's adjoints on their own on both sides of the few-token line, the factors and dX in views
    off their alignment too, against float64 products: f32 sums (few tokens) or two bf16 halves of the
    f32 activations (16 bits) in bf16 products, 2e-5 relative."""
    from r9700training_amd.qlinear import lora_expand_bwd, lora_shrink_bwd

    print(f"case adapter adjoints T={T} C={C} r={r} off={off}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + r)

    def rnd(shape, dtype=torch.float32):
        n = shape[0] * shape[1]
        v = torch.empty(n + 1, dtype=dtype, device="cuda")[int(off):][:n].view(shape)
        return v.copy_(torch.randn(shape, generator=g, device="cuda"))

    X = torch.randn((T, C), generator=g, device="cuda").to(torch.bfloat16)
    A, B = rnd((r, C), torch.bfloat16), rnd((C, r), torch.bfloat16)
    t, u, dX0 = rnd((T, r)), rnd((T, r)), rnd((T, C))
    t_cot, dB = lora_expand_bwd(X, B, 2.0, t=t, t_cot=u.clone())
    dX, dA = lora_shrink_bwd(X, A, t_cot, dX=rnd((T, C)).copy_(dX0), accumulate=True)
    dX2, _ = lora_shrink_bwd(None, A, t_cot, want_dA=False)
    torch.cuda.synchronize()
    x, a, b = X.double(), A.double(), B.double()
    want = u.double() + 2.0 * (x @ b)
    tc = t_cot.double()
    for got, ref in ((t_cot, want), (dB, 2.0 * (x.T @ t.double())), (dX, dX0.double() + tc @ a), (dX2, tc @ a),
                     (dA, tc.T @ x)):
        assert _rel(got, ref) <= 2e-5, _rel(got, ref)


@pytest.mark.parametrize("T,K,r", [(5, 128, 64), (300, 384, 16), (1025, 256, 8)])
def test_shrink_dx_over_its_inputs(T, K, r):
    """The shrink's f32 dX in a buffer that holds t_cot, or A: written after both are read, on either side
    of the few-token line. Against float64 products, with the bound above."""
    from r9700training_amd.qlinear import lora_shrink_bwd

    print(f"case shrink dX over its inputs T={T} K={K} r={r}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    u = torch.randn((T, r), generator=g, device="cuda")
    A = torch.randn((r, K), generator=g, device="cuda").to(torch.bfloat16)
    X = torch.randn((T, K), generator=g, device="cuda").to(torch.bfloat16)
    want = (u.double() @ A.double(), u.double().T @ X.double())
    for over in ("t_cot", "A"):
        dX = torch.empty((max(T, r), K), device="cuda")  # room for A at its start
        at, cot = A, u
        if over == "t_cot":
            cot = dX.view(-1)[: T * r].view(T, r).copy_(u)
        else:
            at = dX.view(torch.bfloat16).view(-1)[: r * K].view(r, K).copy_(A)
        got = lora_shrink_bwd(X, at, cot, dX=dX[:T])
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert _rel(a, b) <= 2e-5, (over, _rel(a, b))


@pytest.mark.parametrize("T,C,r", [(1, 2048, 32), (1, 2176, 32), (255, 5120, 16), (257, 5120, 16), (3, 128, 64)])
def test_expand_one_output(T, C, r):
    """The expand's adjoint asked for t_cot alone (on both sides of its line, 4096 or 2048 columns and 4 a
    token) or dB alone, against float64 products with the bound above; dB alone the bits it has beside t_cot."""
    from r9700training_amd import _ptr, _stream, check, lib
    from r9700training_amd.qlinear import lora_expand_bwd

    print(f"case expand one output T={T} C={C} r={r}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    dY = torch.randn((T, C), generator=g, device="cuda").to(torch.bfloat16)
    B = torch.randn((C, r), generator=g, device="cuda").to(torch.bfloat16)
    t, u = torch.randn((T, r), generator=g, device="cuda"), torch.randn((T, r), generator=g, device="cuda")
    cot, _ = lora_expand_bwd(dY, B, 2.0, t_cot=u.clone(), want_dB=False)
    _, both = lora_expand_bwd(dY, B, 2.0, t=t)
    L = lib()
    ws = torch.empty(L.r97q_lora_expand_bwd_workspace_bytes(T, C, r), dtype=torch.uint8, device="cuda")
    dB = torch.zeros((C, r), device="cuda")
    check(L.r97q_lora_expand_bwd(T, C, _ptr(dY), _ptr(B), r, 2.0, _ptr(t), None, _ptr(dB), _ptr(ws), ws.numel(), _stream()),
          "expand")
    torch.cuda.synchronize()
    assert _rel(cot, u.double() + 2.0 * (dY.double() @ B.double())) <= 2e-5
    assert torch.equal(dB, both) and _rel(dB, 2.0 * (dY.double().T @ t.double())) <= 2e-5


@pytest.mark.parametrize("T,K,r", [(400, 7424, 64), (401, 7552, 64), (1000, 8960, 16), (1008, 8960, 16)])
def test_shrink_dx_alone(T, K, r):
    """The shrink's dX without dA on both sides of its line (3 and 9 million values), against float64
    products with the bound above."""
    from r9700training_amd.qlinear import lora_shrink_bwd

    print(f"case shrink dX alone T={T} K={K} r={r}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    u = torch.randn((T, r), generator=g, device="cuda")
    A = torch.randn((r, K), generator=g, device="cuda").to(torch.bfloat16)
    base = torch.randn((T, K), generator=g, device="cuda")
    dX, _ = lora_shrink_bwd(None, A, u, dX=base.clone(), accumulate=True, want_dA=False)
    torch.cuda.synchronize()
    assert _rel(dX, base.double() + u.double() @ A.double()) <= 2e-5
