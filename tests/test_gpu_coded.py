"""The coded (i8a8h) trunk on the card against the oracle's restatement of the reference's host rows
(src/adjoint/host/linear.cpp:245-317, src/adjoint/host/lora.cpp:246-328): the C entries
r97q_gemm_nt_q_fwd, r97q_gemm_nt_q_dx and r97q_lora_shrink_q_bwd, and the device rows gemm_nt_q
and the coded lora_shrink driven through the registry as the reference's walk drives them.

gemm_nt_q's twin sums each 128-column group exactly (int8 products, int32 sums) and folds the groups
in f32: against the oracle's f64 loop only the f32 fold differs, so its bar is 1e-5 (bf16 Y: the
one rounding of the output, 4e-3).

Bars: gemm_nt_q's code cotangent multiplies a stored IQR weight as bf16(code * scale), one rounding
of each weight (~1.65e-3), so it is held to the base products' 2e-3 relative L2 (a weight carried as
codes + scale through the rows library takes the same single rounding). The shrink's cotangents and
dA carry t_cot as an [hi | lo] bf16 pair and x = code * scale as another: 1e-4."""
import ctypes as C

import numpy as np
import pytest
import torch

import iqr_synth as S
from gpu_util import bf16_tensor, dev, device_desc, f64, host_weight, prepared, rel_l2, stored_operand
from oracle import oracle as O
from test_rows import bf16_round, check, hook, p

pytestmark = pytest.mark.gpu

TOL_BASE = 2e-3
TOL_ADAPTER = 1e-4


def weight_planes(N, K, seed):
    rng = np.random.default_rng(seed)
    return S.trellis(rows=N, cols=K, bits=5, state_bits=16, run_rows=128, rb=1, mad=1, scale_dtype=S.F32,
                     rowf=True, seed=seed, scale_col=(0.75 + 0.5 * rng.random(K // 128)).astype(np.float32))


def codes_and_scales(rng, T, K, groups):
    a = np.rint(rng.uniform(-1.0, 1.0, (T, K)) * 60.0)
    s = (0.02 + 0.05 * rng.random((T, groups))).astype(np.float32).astype(np.float64)
    return a, s


TOL_EXACT = 1e-5


def full_range_codes(rng, T, K):
    """int8 activation codes over the whole range, with per-(row, group) f32 scales."""
    a = rng.integers(-127, 128, (T, K)).astype(np.float64)
    s = (0.01 + 0.05 * rng.random((T, K // 128))).astype(np.float32).astype(np.float64)
    return a, s


@pytest.mark.parametrize("T,N,K", [(300, 256, 384), (512, 384, 256), (64, 128, 1024), (1030, 512, 512), (1, 128, 128),
                                   (257, 640, 896)])
def test_gemm_nt_q_fwd(T, N, K):
    from r9700training_amd.qlinear import gemm_nt_q_fwd

    print(f"case gemm_nt_q_fwd T={T} N={N} K={K}", flush=True)
    rng = np.random.default_rng(7 * T + N + K)
    codes, scale = host_weight(weight_planes(N, K, seed=T + 1))
    cd, scd = dev(codes), dev(scale)
    a, a_scale = full_range_codes(rng, T, K)
    ad = torch.tensor(a.astype(np.int8), device="cuda")
    sd = torch.tensor(a_scale.astype(np.float32), device="cuda")
    got = gemm_nt_q_fwd(cd, scd, ad, sd)
    got_bf = gemm_nt_q_fwd(cd, scd, ad, sd, y_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    want = O.gemm_nt_q_twin(a, a_scale, codes, scale)
    e, e_bf = rel_l2(f64(got), want), rel_l2(f64(got_bf), want)
    print(f"  rel L2 Y {e:.3e} bf16 {e_bf:.3e}", flush=True)
    assert e <= TOL_EXACT and e_bf <= 4e-3
    # the activation scale is applied per group: one group's scale doubled moves the result
    a_scale2 = a_scale.copy()
    a_scale2[:, -1] *= 2.0
    assert rel_l2(f64(got), O.gemm_nt_q_twin(a, a_scale2, codes, scale)) > 10 * TOL_EXACT


def test_gemm_nt_q_fwd_c2():
    """C2's square layer (T = N = K = 4096): the whole Y against the oracle on sampled token rows
    (the first, tile-edge, middle and last), and every row at once through the column sums of the
    group products (each group's sum over m of a * a_scale is one row the oracle multiplies)."""
    from r9700training_amd.qlinear import gemm_nt_q_fwd

    print("case gemm_nt_q_fwd C2", flush=True)
    T = N = K = 4096
    rng = np.random.default_rng(4096)
    sc = (0.75 + 0.5 * rng.random(K // 128)).astype(np.float32)
    planes = S.trellis(rows=N, cols=K, bits=5, state_bits=16, run_rows=256, rb=1, mad=1, scale_dtype=S.F32,
                       rowf=True, seed=11, scale_col=sc, packed=True)
    codes, scale = host_weight(planes)
    a, a_scale = full_range_codes(rng, T, K)
    got = f64(gemm_nt_q_fwd(dev(codes), dev(scale), torch.tensor(a.astype(np.int8), device="cuda"),
                            torch.tensor(a_scale.astype(np.float32), device="cuda")))
    rows = np.unique(np.array([0, 1, 31, 32, 255, 256, 2047, 2048, 3839, 3840, 4094, 4095]))
    e = rel_l2(got[rows], O.gemm_nt_q_twin(a[rows], a_scale[rows], codes, scale))
    # sum over m of Y[m, n] = sum_g (sum_m a[m, g-cols] * a_scale[m, g]) . code[n, g-cols] * scale[n, g]:
    # one f64 row per group, through the oracle with unit activation scales
    x = (a.reshape(T, K // 128, 128) * a_scale[:, :, None]).sum(axis=0).reshape(1, K)
    want_sum = O.gemm_nt_q_twin(x, np.ones((1, K // 128)), codes, scale)[0]
    e_sum = rel_l2(got.sum(axis=0), want_sum)
    print(f"  rel L2 sampled rows {e:.3e} column sums {e_sum:.3e}", flush=True)
    assert e <= TOL_EXACT and e_sum <= TOL_EXACT


def test_gemm_nt_q_fwd_refusals():
    from r9700training_amd import R97qError
    from r9700training_amd.qlinear import gemm_nt_q_fwd

    codes = torch.zeros((128, 300), dtype=torch.int8, device="cuda")
    with pytest.raises(R97qError, match="multiples of 128"):
        gemm_nt_q_fwd(codes, torch.zeros((128, 3), dtype=torch.int16, device="cuda"),
                      torch.zeros((8, 300), dtype=torch.int8, device="cuda"), torch.ones((8, 3), device="cuda"))


@pytest.mark.parametrize("T,N,K", [(300, 256, 384), (512, 384, 256), (64, 128, 1024), (1030, 512, 512)])
def test_gemm_nt_q_dx(T, N, K):
    from r9700training_amd.qlinear import gemm_nt_q_dx

    print(f"case gemm_nt_q_dx T={T} N={N} K={K}", flush=True)
    rng = np.random.default_rng(T + N + K)
    planes = weight_planes(N, K, seed=T)
    keep = []
    w = prepared(planes, keep)
    codes, scale = host_weight(planes)
    dy = bf16_round(rng.standard_normal((T, N)))
    a_scale = (0.02 + 0.05 * rng.random((T, K // 128))).astype(np.float32)
    sd = torch.tensor(a_scale, device="cuda")
    got = gemm_nt_q_dx(w, bf16_tensor(dy), sd)
    base = torch.randn((T, K), dtype=torch.float32, device="cuda")
    acc = gemm_nt_q_dx(w, bf16_tensor(dy), sd, dA=base.clone(), accumulate=True)
    got_bf = gemm_nt_q_dx(w, bf16_tensor(dy), sd, da_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    want = O.gemm_nt_q_adjoint(dy, codes, scale, a_scale.astype(np.float64))
    e, e_acc, e_bf = rel_l2(f64(got), want), rel_l2(f64(acc) - f64(base), want), rel_l2(f64(got_bf), want)
    print(f"  rel L2 dA {e:.3e} accumulate {e_acc:.3e} bf16 {e_bf:.3e}", flush=True)
    assert e <= TOL_BASE and e_acc <= TOL_BASE and e_bf <= 2.6e-3
    # the scale is applied: without it the result is far off
    assert rel_l2(f64(got), O.gemm_nt_adjoint(dy, codes, scale)) > 0.5


@pytest.mark.parametrize("T,K,r,groups", [(300, 256, 16, 2), (512, 384, 8, 3), (200, 256, 64, 1), (128, 512, 32, 4)])
def test_lora_shrink_q_bwd(T, K, r, groups):
    from r9700training_amd.qlinear import lora_shrink_q_bwd

    print(f"case lora_shrink_q_bwd T={T} K={K} r={r} groups={groups}", flush=True)
    rng = np.random.default_rng(T + K + r + groups)
    a, a_scale = codes_and_scales(rng, T, K, groups)
    A = bf16_round(0.05 * rng.standard_normal((r, K)))
    ct = rng.standard_normal((T, r)).astype(np.float32).astype(np.float64)
    da0 = rng.standard_normal((T, K)).astype(np.float32)
    ds0 = rng.standard_normal((T, groups)).astype(np.float32)
    da, ds, dA = lora_shrink_q_bwd(torch.tensor(a.astype(np.int8), device="cuda"),
                                   torch.tensor(a_scale.astype(np.float32), device="cuda"), bf16_tensor(A),
                                   torch.tensor(ct.astype(np.float32), device="cuda"),
                                   da=torch.tensor(da0, device="cuda"), ds=torch.tensor(ds0, device="cuda"))
    torch.cuda.synchronize()
    want_da, want_ds, want_dA = O.lora_shrink_q_adjoint(a, a_scale, np.zeros(T), A.reshape(1, r, K), ct)
    e_da = rel_l2(f64(da) - da0.astype(np.float64), want_da)
    e_ds = rel_l2(f64(ds) - ds0.astype(np.float64), want_ds)
    e_dA = rel_l2(f64(dA), want_dA)
    print(f"  rel L2 da {e_da:.3e} ds {e_ds:.3e} dA {e_dA:.3e}", flush=True)
    assert e_da <= TOL_ADAPTER and e_ds <= TOL_ADAPTER and e_dA <= TOL_ADAPTER


@pytest.mark.parametrize("M,N,K,carried", [(96, 256, 384, False), (200, 512, 256, False), (64, 384, 256, True)])
def test_gemm_nt_q_row(M, N, K, carried):
    print(f"case gemm_nt_q row M={M} N={N} K={K} carried={carried}", flush=True)
    L = hook()
    L.rh_gemm_nt_q.argtypes = [C.c_int64] * 3 + [C.c_void_p] * 7
    rng = np.random.default_rng(M + N + K + 7)
    dy = rng.standard_normal((M, N))
    a_scale = (0.02 + 0.05 * rng.random((M, K // 128))).astype(np.float32).astype(np.float64)
    da0 = rng.standard_normal((M, K))
    da = da0.copy()
    planes = weight_planes(N, K, seed=M + 1)
    codes, scale = host_weight(planes)
    if carried:
        bsc = S.bf16_bits_to_f32(scale).astype(np.float64)
        wc = codes.astype(np.float64)  # held: the call reads it through a raw pointer
        check(L, L.rh_gemm_nt_q(M, N, K, p(dy), p(a_scale), None, None, p(wc), p(bsc), p(da)))
    else:
        keep = []
        enc, raw = stored_operand(planes, keep)
        check(L, L.rh_gemm_nt_q(M, N, K, p(dy), p(a_scale), C.addressof(enc), raw.data_ptr(), None, None, p(da)))
    want = O.gemm_nt_q_adjoint(dy, codes, scale, a_scale, da=da0)
    e = rel_l2(da - da0, want - da0)
    print(f"  rel L2 da {e:.3e}", flush=True)
    assert e <= TOL_BASE


@pytest.mark.parametrize("M,K,R,S_,groups,fused", [(40, 256, 16, 2, 2, False), (33, 384, 8, 1, 3, True),
                                                   (64, 256, 32, 2, 1, True)])
def test_lora_shrink_q_row(M, K, R, S_, groups, fused):
    print(f"case coded lora_shrink row M={M} K={K} R={R} S={S_} groups={groups} fused={fused}", flush=True)
    L = hook()
    L.rh_lora_shrink_q.argtypes = [C.c_int64] * 6 + [C.c_char_p] + [C.c_void_p] * 8 + [C.c_int]
    rng = np.random.default_rng(M + K + R)
    a, a_scale = codes_and_scales(rng, M, K, groups)
    slot = np.array([-1 if m == 1 else (S_ if m == 2 else m % S_) for m in range(M)], np.float64)
    la = bf16_round(0.05 * rng.standard_normal((S_, R, K)))
    ct = rng.standard_normal((M, R)).astype(np.float32).astype(np.float64)
    da0 = rng.standard_normal((M, K))
    ds0 = rng.standard_normal((M, groups))
    da, ds = da0.copy(), ds0.copy()
    dA = np.zeros((S_ * R, K), np.float32)
    group = O.group_width(K, groups)
    check(L, L.rh_lora_shrink_q(M, K, R, S_, groups, group, b"i8", p(a), p(a_scale), p(slot), p(la), p(ct), p(da),
                                p(ds), p(dA), int(fused)))
    want_da, want_ds, want_dA = O.lora_shrink_q_adjoint(a, a_scale, slot, la, ct, da=da0, ds=ds0, fused=True)
    e_da, e_ds, e_dA = rel_l2(da - da0, want_da - da0), rel_l2(ds - ds0, want_ds - ds0), rel_l2(dA, want_dA)
    print(f"  rel L2 da {e_da:.3e} ds {e_ds:.3e} dA {e_dA:.3e}", flush=True)
    assert e_da <= TOL_ADAPTER and e_ds <= TOL_ADAPTER and e_dA <= TOL_ADAPTER
    # base rows (1: slot -1, 2: past the pool) get nothing
    assert np.array_equal(da[1:3], da0[1:3]) and np.array_equal(ds[1:3], ds0[1:3])


def test_coded_entry_refusals():
    """The C entry serves K a multiple of 128 (the rows pad other widths) and a group width whose
    groups fit K; it refuses the rest by name."""
    from r9700training_amd import R97qError
    from r9700training_amd.qlinear import lora_shrink_q_bwd

    with pytest.raises(R97qError, match="K a multiple of 128"):
        lora_shrink_q_bwd(torch.zeros((8, 300), dtype=torch.int8, device="cuda"),
                          torch.ones((8, 3), device="cuda"), torch.zeros((16, 300), dtype=torch.bfloat16, device="cuda"),
                          torch.zeros((8, 16), device="cuda"))
    with pytest.raises(R97qError, match="do not fit K"):
        lora_shrink_q_bwd(torch.zeros((8, 256), dtype=torch.int8, device="cuda"),
                          torch.ones((8, 3), device="cuda"), torch.zeros((16, 256), dtype=torch.bfloat16, device="cuda"),
                          torch.zeros((8, 16), device="cuda"), group_width=128)


@pytest.mark.parametrize("T,K,gw,r", [(5, 128, 64, 8), (33, 384, 128, 16), (200, 768, 256, 64), (70, 1152, 128, 32),
                                      (129, 1024, 512, 16), (64, 896, 96, 16), (1, 640, 128, 64), (700, 256, 64, 64)])
def test_int8_codes_match_the_general_path(T, K, gw, r):
    """The coded shrink's adjoint over int8 codes with group widths the fused kernels take (64, 128, 256
    columns; a multiple of 256 for dA) and others, against the same codes handed over as f32 values,
    which take the general path: the two hold the f32 operands as two bf16 halves each (16 bits), the
    general one the activation's value, the fused one the scaled cotangent -- 2e-5 relative."""
    from r9700training_amd.qlinear import lora_shrink_q_bwd

    print(f"case coded shrink T={T} K={K} gw={gw} r={r}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + K)
    groups = (K + gw - 1) // gw
    code = torch.randint(-128, 128, (T, K), generator=g, device="cuda", dtype=torch.int8)
    s = 0.01 + torch.rand((T, groups), generator=g, device="cuda")
    A = (0.1 * torch.randn((r, K), generator=g, device="cuda")).to(torch.bfloat16)
    t = torch.randn((T, r), generator=g, device="cuda")
    base = [torch.randn(sh, generator=g, device="cuda") for sh in ((T, K), (T, groups), (r, K))]
    out = [lora_shrink_q_bwd(a, s, A, t, da=base[0].clone(), ds=base[1].clone(), dA=base[2].clone(), group_width=gw)
           for a in (code, code.float(), code)]
    only = lora_shrink_q_bwd(code, s, A, t, ds=base[1].clone(), want=("ds",), group_width=gw)
    torch.cuda.synchronize()
    for i, (a, b, c) in enumerate(zip(*out)):
        assert torch.equal(a, c), i
        d = (b - base[i]).double()
        assert float((a.double() - b.double()).norm() / d.norm()) <= 2e-5, i
    assert torch.equal(only[1], out[0][1])


@pytest.mark.parametrize("T,K,gw,r", [(5, 128, 64, 8), (200, 768, 256, 64), (129, 1024, 512, 16), (64, 896, 96, 16)])
def test_coded_shrink_da_over_t_cot(T, K, gw, r):
    """da added into the buffer that holds t_cot: t_cot is read first, whichever kernels the group width
    takes -- the separate buffers' bits, plus t_cot."""
    from r9700training_amd.qlinear import lora_shrink_q_bwd

    print(f"case coded shrink da over t_cot T={T} K={K} gw={gw} r={r}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + K)
    groups = (K + gw - 1) // gw
    code = torch.randint(-128, 128, (T, K), generator=g, device="cuda", dtype=torch.int8)
    s = 0.01 + torch.rand((T, groups), generator=g, device="cuda")
    A = (0.1 * torch.randn((r, K), generator=g, device="cuda")).to(torch.bfloat16)
    t = torch.randn((T, r), generator=g, device="cuda")
    base = torch.zeros(T * K, device="cuda")
    base[: T * r] = t.view(-1)
    want = lora_shrink_q_bwd(code, s, A, t, da=base.clone().view(T, K), group_width=gw)
    da = base.clone()
    got = lora_shrink_q_bwd(code, s, A, da[: T * r].view(T, r), da=da.view(T, K), group_width=gw)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i


@pytest.mark.parametrize("T,N,K,bf16", [(1, 128, 128, False), (31, 256, 640, True), (33, 384, 1152, False),
                                        (100, 8192, 128, False), (130, 6528, 256, False), (129, 128, 4224, False),
                                        (32, 4096, 128, False), (64, 4096, 256, True), (65, 4096, 256, False),
                                        (100, 8192, 1024, False), (129, 8192, 1024, False)])
def test_coded_forward_few_tokens(T, N, K, bf16):
    """The coded forward on both sides of its few-token line (128 tiles of 32 x 32 a group, up to 1024: 32 x
    4096 over one, 64 x 4096 over two and 100 x 8192 over eight the last of it) and off 16 bytes, against
    float64: the group sums are exact, so what is left is the f32 fold over the groups (1e-6 relative) and a bf16 output's rounding."""
    from r9700training_amd.qlinear import gemm_nt_q_fwd

    print(f"case coded forward T={T} N={N} K={K} bf16={bf16}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T * N + K)

    def codes(rows):
        return torch.randint(-127, 128, (rows, K), generator=g, device="cuda", dtype=torch.int8)

    w, a = codes(N), codes(T)
    ws = (0.001 + 0.01 * torch.rand((N, K // 128), generator=g, device="cuda")).to(torch.bfloat16)
    s = 0.01 + torch.rand((T, K // 128), generator=g, device="cuda")
    off = torch.empty(T * K + 1, dtype=torch.int8, device="cuda")[1:].view(T, K).copy_(a)
    wide = lambda c, x: c.double() * x.double().repeat_interleave(128, 1)  # noqa: E731
    ref = wide(a, s) @ wide(w, ws).T
    dt = torch.bfloat16 if bf16 else torch.float32
    for x in (a, off):
        Y = gemm_nt_q_fwd(w, ws, x, s, y_dtype=dt)
        torch.cuda.synchronize()
        assert float((Y.double() - ref).norm() / ref.norm()) <= (2.5e-3 if bf16 else 1e-6)


@pytest.mark.parametrize("T,N,K,bits", [(1, 128, 128, 5), (32, 384, 256, 3), (33, 256, 512, 8), (64, 640, 384, 4),
                                        (65, 256, 1024, 6), (257, 128, 16384, 5), (513, 256, 16384, 8),
                                        (1200, 128, 8192, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_coded_dx_tiles(T, N, K, bits, dtype):
    """gemm_nt_q's adjoint over its token tiles (32, 64, 128, 256 and 512 tokens), written and added to,
    against the plain dX product's f32 output times the scale: the same bf16 products, so the order of
    the f32 sums (1e-6) and a bf16 output's roundings are all that differ."""
    from r9700training_amd import R97Q_DECODE_AUTO, R97Q_DECODE_FUSED, lib
    from r9700training_amd.qlinear import QWeight, gemm_nt_q_dx, qlinear_lora_bwd
    from gpu_util import device_desc

    print(f"case coded dX T={T} N={N} K={K} bits={bits} {dtype}", flush=True)
    keep = []
    p = S.trellis(rows=N, cols=K, bits=5 if bits == 8 else bits, run_rows=128, rowf=True, seed=T, packed=True,
                  scale_col=np.ones(K // 128, np.float32))
    sc = torch.ones(K // 128, device="cuda")
    w = QWeight(device_desc(p, keep), scale_col=sc, codes8=bits == 8)
    g = torch.Generator(device="cuda").manual_seed(T + N)
    dY = torch.randn((T, N), generator=g, device="cuda").to(torch.bfloat16)
    s = 0.01 + torch.rand((T, K // 128), generator=g, device="cuda")
    lib().r97q_set_decode_once(R97Q_DECODE_FUSED)
    try:
        plain, _, _ = qlinear_lora_bwd(w, None, dY, dx_dtype=torch.float32)
    finally:
        lib().r97q_set_decode_once(R97Q_DECODE_AUTO)
    want = plain.double() * s.double().repeat_interleave(128, 1)
    base = torch.randn((T, K), generator=g, device="cuda").to(dtype)
    got = gemm_nt_q_dx(w, dY, s, da_dtype=dtype)
    added = gemm_nt_q_dx(w, dY, s, dA=base.clone(), accumulate=True)
    torch.cuda.synchronize()
    tol = 1e-6 if dtype == torch.float32 else 2.5e-3
    assert float((got.double() - want).norm() / want.norm()) <= tol
    both = want + base.double()
    assert float((added.double() - both).norm() / both.norm()) <= tol
