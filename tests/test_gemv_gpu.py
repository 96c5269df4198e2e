"""The HIP GEMV / skinny GEMM against the oracle (the reference's ``tests/kernels/test_gemv_T.py`` strategy):

* dequantized weights decoded by the kernels' own decode path are bit-identical to the oracle's ``dequantize``
  (all four formats, including every E4M3 block-scale code and every finite FP8 code, signed zero included);
* ``y = x·Wᵀ`` within the reference's leaf gate (``OracleCheck.ok``: ≤ 2 BF16 ULP at the output RMS, relative error
  < 1e-4) against a float64 matmul of the exact dequantized matrix, for M = 1, 2, 8, 16, ragged N, the residual and
  silu·mul epilogues (rounded chains gated by ``ok_rounded``) and the fused input RMSNorm;
* the BASELINE shapes (INT4 4096×4096, NVFP4 17408×5120 and 5120×17408 at M = 1 and 8).
"""

import numpy as np
import pytest

from helpers import from_dev_bf16, spec_of, to_dev_bf16
from oracle import formats as OF
from oracle import nn as ON
from oracle.fp import rbf
from oracle.gates import check_against_oracle

pytestmark = pytest.mark.gpu


def _matrix(fmt, n, k, rng):
    if fmt == "nvfp4":
        return OF.nvfp4_random(n, k, rng)
    if fmt == "fp8_e4m3":
        return OF.fp8_random(n, k, rng)
    if fmt == "int4_affine":
        return OF.int4_random(n, k, rng)
    from oracle.fp import f32_to_bf16
    return {"format": "bf16", "weight": f32_to_bf16((rng.standard_normal((n, k)) * 0.02).astype(np.float32))}


def _dequant(m):
    if m["format"] == "bf16":
        from oracle.fp import bf16_to_f32
        return bf16_to_f32(m["weight"])
    return OF.dequantize(m)


def _upload(torch, m):
    from monolith_mi355 import kernels
    return kernels.upload(spec_of(m))


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "bf16", "fp8_e4m3"])
@pytest.mark.parametrize("n,k", [(16, 128), (37, 512), (300, 1024)])
def test_dequant_bit_exact(torch_gpu, fmt, n, k, rng):
    from monolith_mi355 import kernels
    if fmt == "bf16" and k % 32:
        pytest.skip()
    m = _matrix(fmt, n, k, rng)
    w = _upload(torch_gpu, m)
    got = kernels.dequant(w).cpu().numpy()
    ref = _dequant(m)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


def test_dequant_every_scale_code(torch_gpu, rng):
    """All 126 finite non-negative E4M3 block-scale codes and all 16 E2M1 codes, bit for bit
    (the reference's tests/kernels/test_nvfp4_scale_decode.py:11-27)."""
    from monolith_mi355 import kernels
    n, k = 128, 256
    m = OF.nvfp4_random(n, k, rng)
    codes = np.arange(n * k // 16) % 0x7F                      # 0x00..0x7E cycling
    m["weight_scale"] = codes.astype(np.uint8).reshape(n, k // 16)
    m["weight"] = (np.arange(n * k // 2) % 256).astype(np.uint8).reshape(n, k // 2)
    got = kernels.dequant(_upload(torch_gpu, m)).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), OF.nvfp4_dequantize(m).view(np.uint32))


def _plan(w, x, **kw):
    """The launch plan (``mi_gemv_plan``) of this GEMV."""
    import ctypes as C
    from monolith_mi355 import kernels
    from monolith_mi355.runtime import hip
    d, _ = kernels._gemv_desc(w, x, **kw)
    out = (C.c_int32 * 7)()
    hip.call("mi_gemv_plan", C.byref(d), out)
    return list(out)


def _run(torch, m, x, **kw):
    """FP32 output, as the reference's gemv_T test reads it (tests/kernels/test_gemv_T.py:21-46)."""
    from monolith_mi355 import kernels
    w = _upload(torch, m)
    y = kernels.gemv(w, to_dev_bf16(torch, x), out_f32=True, **kw)
    torch.cuda.synchronize()
    return y.cpu().numpy()


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "bf16", "fp8_e4m3"])
@pytest.mark.parametrize("mtok", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("n,k", [(48, 256), (77, 1024), (1040, 2048)])
def test_gemv_matches_oracle(torch_gpu, fmt, mtok, n, k, rng):
    m = _matrix(fmt, n, k, rng)
    x = rbf(rng.standard_normal((mtok, k)).astype(np.float32))
    got = _run(torch_gpu, m, x)
    ref = ON.matmul_acc(x, _dequant(m))
    chk = check_against_oracle(got, ref)
    assert chk.ok() and chk.within, (fmt, mtok, n, k, chk)
    from monolith_mi355 import kernels                      # the BF16 output is the same number rounded once
    yb = from_dev_bf16(kernels.gemv(_upload(torch_gpu, m), to_dev_bf16(torch_gpu, x)))
    assert np.array_equal(yb, rbf(got))


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3"])
@pytest.mark.parametrize("mtok", [1, 8])
def test_gemv_residual(torch_gpu, fmt, mtok, rng):
    n, k = 160, 1024
    m = _matrix(fmt, n, k, rng)
    x = rbf(rng.standard_normal((mtok, k)))
    res = rbf(rng.standard_normal((mtok, n)))
    from monolith_mi355 import kernels
    w = _upload(torch_gpu, m)
    y = kernels.gemv(w, to_dev_bf16(torch_gpu, x), epilogue="residual", residual=to_dev_bf16(torch_gpu, res))
    got = from_dev_bf16(y)
    ref = ON.linear(x, _dequant(m), epilogue="residual", residual=res)
    chk = check_against_oracle(got, ref)
    assert chk.ok_rounded() and chk.within and chk.max_ulp_elementwise <= 1, chk


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3"])
@pytest.mark.parametrize("rounded", [False, True])
@pytest.mark.parametrize("mtok", [1, 8])
def test_gemv_silu_mul(torch_gpu, fmt, rounded, mtok, rng):
    inter, k = 96, 512
    gate, up = _matrix(fmt, inter, k, rng), _matrix(fmt, inter, k, rng)
    if fmt == "nvfp4":
        up["weight_scale_2"] = gate["weight_scale_2"] * 1.5              # distinct tensor scales per part
    if fmt == "fp8_e4m3":
        up["weight_scale"] = gate["weight_scale"] * 1.5
    slab = OF.stack_rows([gate, up])
    perm = ON.interleave_chunks(inter, inter, 8)
    slab = OF.permute_rows(slab, perm)
    from monolith_mi355 import kernels
    from monolith_mi355.formats import DequantSpec
    spec = spec_of(dict(slab, weight_scale=1.0) if fmt == "fp8_e4m3" else dict(slab, weight_scale_2=1.0))
    w = kernels.upload(spec, row_scales=[slab["row_scale"]] if fmt in ("nvfp4", "fp8_e4m3") else None)
    x = rbf(rng.standard_normal((mtok, k)))
    epi = "silu_mul_rounded" if rounded else "silu_mul"
    got = from_dev_bf16(kernels.gemv(w, to_dev_bf16(torch_gpu, x), epilogue=epi))
    wg, wu = OF.dequantize(gate), OF.dequantize(up)
    ref = ON.linear(x, np.concatenate([wg, wu]), epilogue="silu_mul", round_silu=rounded)
    chk = check_against_oracle(got, ref)
    assert got.shape == (mtok, inter)
    assert chk.ok_rounded() and chk.within, chk


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "bf16", "fp8_e4m3"])
@pytest.mark.parametrize("mtok", [1, 8])
def test_gemv_fused_norm(torch_gpu, fmt, mtok, rng):
    n, k = 200, 2048
    m = _matrix(fmt, n, k, rng)
    h = rbf(rng.standard_normal((mtok, k)) * 3)
    wn = rbf(rng.standard_normal(k) * 0.2)
    nw = (1.0 + wn).astype(np.float32)
    from monolith_mi355 import kernels
    w = _upload(torch_gpu, m)
    got = kernels.gemv(w, to_dev_bf16(torch_gpu, h), norm_w=torch_gpu.from_numpy(nw).cuda(), eps=1e-6,
                       out_f32=True).cpu().numpy()
    xn = ON.rms_norm(h, wn, 1e-6)
    ref = ON.matmul_acc(xn, _dequant(m))
    chk = check_against_oracle(got, ref)
    assert chk.ok_rounded() and chk.within, chk


@pytest.mark.parametrize("fmt,n,k,mtok", [("int4_affine", 4096, 4096, 1), ("nvfp4", 17408, 5120, 1),
                                          ("nvfp4", 17408, 5120, 8), ("nvfp4", 5120, 17408, 1),
                                          ("nvfp4", 5120, 17408, 8)])
def test_gemv_baseline_shapes(torch_gpu, fmt, n, k, mtok):
    rng = np.random.default_rng(n + k + mtok)
    m = _matrix(fmt, n, k, rng)
    x = rbf(rng.standard_normal((mtok, k)))
    got = _run(torch_gpu, m, x)
    w = _dequant(m)
    ref = ON.matmul_acc(x, w)
    chk = check_against_oracle(got, ref)
    assert chk.ok() and chk.within, chk


def test_gemv_repeat_is_bit_identical(torch_gpu, rng):
    """Split-K partials are combined in a fixed order: two runs give the same bits."""
    from monolith_mi355 import kernels
    m = _matrix("nvfp4", 5120, 17408, rng)
    w = _upload(torch_gpu, m)
    x = to_dev_bf16(torch_gpu, rbf(rng.standard_normal((8, 17408))))
    a = kernels.gemv(w, x).clone()
    b = kernels.gemv(w, x)
    assert torch_gpu.equal(a, b)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "bf16", "fp8_e4m3"])
@pytest.mark.parametrize("n,k", [(1040, 2048), (336, 1664)])
@pytest.mark.parametrize("epi", [None, "residual", "silu_mul"])
def test_gemv_tiles_per_workgroup(torch_gpu, fmt, n, k, epi, rng, monkeypatch):
    """M = 1 with a workgroup streaming 1..5 tiles (the fused-norm plan): every tile's K slices are added in the
    same order, so the output is bit-identical to one tile per workgroup, and within the oracle bar."""
    from monolith_mi355 import kernels
    if epi == "silu_mul":
        n = n // 16 * 16
    m = _matrix(fmt, n, k, rng)
    w = _upload(torch_gpu, m)
    h = rbf(rng.standard_normal((1, k)) * 3)
    wn = rbf(rng.standard_normal(k) * 0.2)
    nw = torch_gpu.from_numpy((1.0 + wn).astype(np.float32)).cuda()
    res = rbf(rng.standard_normal((1, n)))
    kw = dict(norm_w=nw, eps=1e-6, epilogue=epi)
    if epi == "residual":
        kw["residual"] = to_dev_bf16(torch_gpu, res)
    outs = {}
    for rt in (1, 2, 3, 5):
        monkeypatch.setenv("MI_GEMV_ROW", f"4,1,{rt}")
        outs[rt] = from_dev_bf16(kernels.gemv(w, to_dev_bf16(torch_gpu, h), **kw))
    monkeypatch.delenv("MI_GEMV_ROW")
    for rt in (2, 3, 5):
        assert np.array_equal(outs[rt].view(np.uint16), outs[1].view(np.uint16)), rt
    xn = ON.rms_norm(h, wn, 1e-6)
    wd = _dequant(m)
    if epi == "silu_mul":
        ref = ON.linear(xn, wd[np.argsort(ON.interleave_chunks(n // 2, n // 2, 8))], epilogue="silu_mul")
    else:
        ref = ON.linear(xn, wd, epilogue=epi, residual=res if epi else None)
    chk = check_against_oracle(outs[1], ref)
    assert chk.ok_rounded() and chk.within, chk


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine"])
@pytest.mark.parametrize("mtok", [1, 2, 3, 8, 16])
@pytest.mark.parametrize("plan", [None, "4,3", "tk", "rowm2"])
def test_gemv_gated_head_norm(torch_gpu, fmt, mtok, plan, rng, monkeypatch):
    """The Gated DeltaNet output norm fused into the output projection's input staging: per 128-column head,
    bf16(bf16(bf16(w)·bf16(o·r))·silu(z)), then the GEMV — against the oracle's gated_rms_norm and matmul (M ≥ 3:
    gemv_tk, whatever gemv_rowm split is asked for)."""
    from monolith_mi355 import kernels
    if plan == "tk":
        monkeypatch.setenv("MI_GEMV_KERNEL", "tk")
    elif plan == "rowm2":
        monkeypatch.setenv("MI_GEMV_ROWM", "2,0")
    elif plan:
        monkeypatch.setenv("MI_GEMV_ROW", plan)
    heads, n = 12, 320
    k = heads * 128
    m = _matrix(fmt, n, k, rng)
    o = rbf(rng.standard_normal((mtok, k)) * 0.3)
    zfull = rbf(rng.standard_normal((mtok, k + 64)) * 2)       # z as a view with its own row stride
    wn = rbf(1 + rng.standard_normal(128) * 0.2).astype(np.float32)
    zd = to_dev_bf16(torch_gpu, zfull)[:, 32: 32 + k]
    got = kernels.gemv(_upload(torch_gpu, m), to_dev_bf16(torch_gpu, o), out_f32=True,
                       gated_norm=(torch_gpu.from_numpy(wn).cuda(), zd, 1e-6)).cpu().numpy()
    xn = ON.gated_rms_norm(o.reshape(mtok, heads, 128), zfull[:, 32: 32 + k].reshape(mtok, heads, 128), wn, 1e-6)
    ref = ON.matmul_acc(xn.reshape(mtok, k), _dequant(m))
    chk = check_against_oracle(got, ref)
    assert chk.ok_rounded() and chk.within, (fmt, mtok, plan, chk)


@pytest.mark.parametrize("fmt", ["nvfp4", "fp8_e4m3", "int4_affine", "bf16"])
@pytest.mark.parametrize("mtok", [3, 8, 16])
@pytest.mark.parametrize("n,k,plan", [(1040, 2048, None), (1040, 2048, "1,3"), (336, 6144, "2,1"),
                                      (336, 6144, "3,2"), (5120, 17408, None)])
@pytest.mark.parametrize("epi", [None, "residual", "silu_mul"])
def test_gemv_rowm_plans(torch_gpu, fmt, mtok, n, k, plan, epi, rng, monkeypatch):
    """The M >= 3 kernel (K slices per wave on the matrix cores, several tiles per workgroup) over
    forced K splits and tiles per workgroup, against the oracle."""
    from monolith_mi355 import kernels
    if plan:
        monkeypatch.setenv("MI_GEMV_ROWM", plan)
    m = _matrix(fmt, n, k, rng)
    x = rbf(rng.standard_normal((mtok, k)))
    res = rbf(rng.standard_normal((mtok, n)))
    kw = dict(epilogue=epi)
    if epi == "residual":
        kw["residual"] = to_dev_bf16(torch_gpu, res)
    w, xd = _upload(torch_gpu, m), to_dev_bf16(torch_gpu, x)
    launch = _plan(w, xd, **kw)
    assert launch[0] == 3 and (not plan or plan[0] == "1" or launch[4] == int(plan[0])), launch
    got = from_dev_bf16(kernels.gemv(w, xd, **kw))
    wd = _dequant(m)
    if epi == "silu_mul":
        ref = ON.linear(x, wd[np.argsort(ON.interleave_chunks(n // 2, n // 2, 8))], epilogue="silu_mul")
    else:
        ref = ON.linear(x, wd, epilogue=epi, residual=res if epi else None)
    chk = check_against_oracle(got, ref)
    assert chk.ok_rounded() and chk.within, (mtok, n, k, plan, epi, chk)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("mtok,n", [(2, 8192), (3, 1040), (8, 1040), (16, 1040)])
@pytest.mark.parametrize("spread", [0.0, 2.0])
def test_gemv_rowm_sums_in_32_bits(torch_gpu, fmt, mtok, n, spread, rng, monkeypatch):
    """The FP32 output against 64 bits, on the matrix cores' default routes, for normal activations and ones over several
    binades (exp(2 N)). A value goes through about thirty FP32 additions (16 MFMA steps or groups of a slice, ten slices)
    of sums of up to about twice the result: sqrt(30) roundings of 0.29·2^-23 each come to 2^-21.6 of twice the result's
    norm at most, an operand that loses bits on the way to far more. Nor is it more than
    1.25 times the error of the kernel that took such calls before (gemv_row, gemv_tk), whose own spread over thousands of
    outputs is a few percent."""
    torch, k = torch_gpu, 5120
    w = _upload(torch, _matrix(fmt, n, k, rng))
    from monolith_mi355 import kernels
    x = rng.standard_normal((mtok, k)) * np.exp(spread * rng.standard_normal((mtok, k)))
    xd = to_dev_bf16(torch, rbf(x.astype(np.float32)))
    assert _plan(w, xd)[0] == 3
    ref = xd.double().cpu() @ kernels.dequant(w).double().cpu().T

    def error():
        return ((kernels.gemv(w, xd, out_f32=True).double().cpu() - ref).norm() / ref.norm()).item()

    err = error()
    assert err <= 2.0 ** -21.6, err
    if mtok == 2 or fmt != "fp8_e4m3":
        monkeypatch.setenv("MI_GEMV_KERNEL", "row" if mtok == 2 else "tk")
        assert _plan(w, xd)[0] == (1 if mtok == 2 else 2)
        before = error()
        print(f"{fmt} M={mtok} spread={spread}: {err:.2e}, before {before:.2e}", flush=True)
        assert err <= 1.25 * before, (err, before)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("mtok", [3, 4, 5, 8, 9, 13, 16])
@pytest.mark.parametrize("n,k", [(24, 128), (4117, 640), (56, 896), (33, 1792), (40, 6656)])
def test_gemv_rowm_edges(torch_gpu, fmt, mtok, n, k, rng):
    """Every remainder of the four rows staged at a time, a slice of one chunk, two K splits, one tile a workgroup (NVFP4
    under a slice of K runs on gemv_tk, small BF16 in token passes on gemv_row); a row of zeros, one scaled by 2^60 and
    one by 2^-60 (each row's own power-of-two prescale): every row inside the leaf gate of its own values."""
    m = _matrix(fmt, n, k, rng)
    launch = _plan(_upload(torch_gpu, m), to_dev_bf16(torch_gpu, np.zeros((mtok, k), np.float32)))
    assert launch[0] == (2 if fmt == "nvfp4" and k < 512 else 1 if fmt == "bf16" and n * k * 2 <= 256 << 10 else 3)
    x = rbf(rng.standard_normal((mtok, k)).astype(np.float32))
    x[0] = 0.0
    x[1] *= 2.0 ** 60
    x[mtok - 1] *= 2.0 ** -60
    got = _run(torch_gpu, m, x)
    ref = ON.matmul_acc(x, _dequant(m))
    assert not got[0].any()
    for i in range(1, mtok):
        e = (0, 60)[i == 1] or (0, -60)[i == mtok - 1]
        chk = check_against_oracle(got[i: i + 1] * np.float32(2.0 ** -e), ref[i: i + 1] * np.float32(2.0 ** -e))
        assert chk.ok() and chk.within, (fmt, mtok, n, k, i, chk)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("mtok", [3, 8, 13])
def test_gemv_rowm_tiles_per_workgroup(torch_gpu, fmt, mtok, rng, monkeypatch):
    """67 tiles as 1 to 9 a workgroup, an uneven last round in each: every tail of the loop with two tiles in flight and
    of the one with one, and the activation stage reused for the partials: the bits of one tile a workgroup, which lie
    inside the leaf gate."""
    from monolith_mi355 import kernels
    n, k = 1067, 1152
    m = _matrix(fmt, n, k, rng)
    x = rbf(rng.standard_normal((mtok, k)).astype(np.float32))
    w, xd = _upload(torch_gpu, m), to_dev_bf16(torch_gpu, x)
    outs = {}
    for rt in (1, 2, 3, 4, 5, 7, 9):
        monkeypatch.setenv("MI_GEMV_ROWM", f"0,{rt}")
        launch = _plan(w, xd)
        assert launch[0] == 3 and launch[3] == rt, launch
        outs[rt] = kernels.gemv(w, xd, out_f32=True).cpu().numpy()
        assert np.array_equal(outs[rt].view(np.uint32), outs[1].view(np.uint32)), rt
    chk = check_against_oracle(outs[1], ON.matmul_acc(x, _dequant(m)))
    assert chk.ok() and chk.within, (fmt, mtok, chk)


@pytest.mark.parametrize("fmt,n,k", [("fp8_e4m3", 170056, 2048), ("nvfp4", 170056, 2048), ("fp8_e4m3", 57352, 6144)])
def test_gemv_rowm_tall(torch_gpu, fmt, n, k):
    """A matrix of more tiles than one round of workgroups holds partials of (the last tile half full): every row of
    the product against the decoded matrix in float64. The packed bytes are random (any are codes of the format; the
    decode itself is pinned elsewhere)."""
    from monolith_mi355 import kernels
    from monolith_mi355.formats.pack import pack_bytes
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    data = torch.randint(0, 256, (pack_bytes(fmt, n, k),), dtype=torch.uint8, generator=g, device="cuda")
    data &= 0xF7 if fmt == "fp8_e4m3" else 0x7F                          # no NaN code / NVFP4 scale
    if fmt == "nvfp4":
        data &= 0xBF                                                     # scales below 2
    w = kernels.PackedWeight(fmt, n, k, 1, data, torch.rand((n + 15) // 16 * 16, generator=g, device="cuda"))
    x = torch.randn(5, k, generator=g, device="cuda").to(torch.bfloat16)
    plan = _plan(w, x)
    assert plan[0] == 3 and plan[3] * plan[1] * 1024 <= 160 * 1024 and plan[6] > 256, plan
    got = kernels.gemv(w, x, out_f32=True)
    wd = kernels.dequant(w)
    for lo in range(0, n, 32768):
        part = wd[lo: lo + 32768].double()
        ref = x.double() @ part.T
        bound = x.double().abs() @ part.abs().T          # 32-bit sums of k products: a part of sum |x·w|
        assert ((got[:, lo: lo + 32768].double() - ref).abs() <= 2.0 ** -18 * bound).all(), (fmt, lo)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("mtok", [2, 3, 8])
def test_gemv_rowm_small_beside_large(torch_gpu, fmt, mtok, rng):
    """One value of a 512-column slice 2^30 above the others, on a zero weight: the small ones keep all their bits (eight,
    with F16's 24 below the slice's maximum), so the rest of the sum is a 32-bit sum."""
    _small_beside_large(torch_gpu, fmt, mtok, (-30,), rng)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
def test_gemv_two_tokens_any_range(torch_gpu, fmt, rng):
    """Two tokens keep every activation exact, however far below its slice's maximum (their operand rows are there for
    it): 32 binades are one operand, 200 seven of them."""
    _small_beside_large(torch_gpu, fmt, 2, (-31, -32, -60, -100, -200), rng)


def _small_beside_large(torch, fmt, mtok, exps, rng):
    from monolith_mi355 import kernels
    k, big = 3072, 1000
    block = _matrix(fmt, 96, k, rng)
    block["weight"][:, big // 2 if fmt in ("nvfp4", "int4_affine") else big] = 0
    if fmt == "int4_affine":                                  # code 0 without an offset in its group
        block["biases"][:, big // 64] = 0
    wd = _dequant(block).astype(np.float64)
    assert not wd[:, big].any()
    per_row = {"nvfp4": 1728, "int4_affine": 1728, "fp8_e4m3": 3072, "bf16": 6144}[fmt]
    rep = 1 if mtok > 2 else -(-((40 if fmt == "fp8_e4m3" else 20) << 20) // (per_row * 96)) + 1
    m = {kk: (np.tile(v, (rep, 1)) if isinstance(v, np.ndarray) and v.ndim == 2 else v) for kk, v in block.items()}
    w = _upload(torch, m)
    for exp in exps:
        x = rbf((1 + rng.random((mtok, k))) * np.where(rng.random((mtok, k)) < 0.5, -1, 1))
        up = min(0, exp + 110)                                # the small ones stay above 2^-110
        x = rbf(x * np.float32(2.0 ** (exp - up)))
        x[:, big] = rbf(np.float32(1.5 * 2.0 ** -up))
        xd = to_dev_bf16(torch, x)
        assert _plan(w, xd)[0] == 3
        got = kernels.gemv(w, xd, out_f32=True).cpu().numpy().astype(np.float64)
        ref = np.tile(x.astype(np.float64) @ wd.T, (1, rep))
        bound = np.tile(np.abs(x.astype(np.float64)) @ np.abs(wd).T, (1, rep))
        assert (np.abs(got - ref) <= 2.0 ** -18 * bound).all(), (fmt, mtok, exp)
        if mtok == 2:                                         # the second token alone, the first of ordinary values
            x[0] = rbf(rng.standard_normal(k).astype(np.float32))
            got = kernels.gemv(w, to_dev_bf16(torch, x), out_f32=True).cpu().numpy().astype(np.float64)
            ref = np.tile(x.astype(np.float64) @ wd.T, (1, rep))
            bound = np.tile(np.abs(x.astype(np.float64)) @ np.abs(wd).T, (1, rep))
            assert (np.abs(got - ref) <= 2.0 ** -18 * bound).all(), (fmt, exp)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("mtok", [2, 3, 8])
@pytest.mark.parametrize("high", [False, True])
def test_gemv_rowm_extreme_rows(torch_gpu, fmt, mtok, high, rng):
    """Rows at the ends of the BF16 range keep their values on the matrix cores: one scaled by 2^120 (INT4's 2^24 on top
    of the row's power is past FP32 from 2^118 on; NVFP4 and FP8 by 2^112: the sum of their unscaled codes has to stay in
    FP32) or by 2^-120 (below 2^-112 the prescale's own exponent is past it), one of zeros but for a
    subnormal, beside ordinary ones. The scaled row inside the leaf gate; the subnormal one, whose products FP32 holds only
    as subnormals, within its smallest normal number."""
    from monolith_mi355 import kernels
    torch = torch_gpu
    k = 3072
    exp = -120 if not high else 112 if fmt in ("nvfp4", "fp8_e4m3") else 120
    block = _matrix(fmt, 96, k, rng)
    per_row = {"nvfp4": 1728, "int4_affine": 1728, "fp8_e4m3": 3072, "bf16": 6144}[fmt]
    # two tokens: enough rows (the block again and again) for gemv_rowm
    rep = 1 if mtok > 2 else -(-((40 if fmt == "fp8_e4m3" else 20) << 20) // (per_row * 96)) + 1
    m = {kk: (np.tile(v, (rep, 1)) if isinstance(v, np.ndarray) and v.ndim == 2 else v) for kk, v in block.items()}
    w = _upload(torch, m)
    x = rbf(rng.standard_normal((mtok, k)).astype(np.float32))
    x[1] *= np.float32(2.0 ** exp)
    x[1] = rbf(x[1])
    x[0, :512] = 0.0
    x[0, 100] = np.float32(2.0 ** -130)
    only = np.zeros_like(x)
    only[:, 0] = x[:, 0]
    only[0, 0], only[0, 700] = 0.0, np.float32(2.0 ** -130)
    for xi in (x, only):
        xd = to_dev_bf16(torch, xi)
        assert _plan(w, xd)[0] == 3
        got = kernels.gemv(w, xd, out_f32=True).cpu().numpy()
        assert np.count_nonzero(~np.isfinite(got)) == 0
        ref = np.tile(ON.matmul_acc(xi.astype(np.float64), _dequant(block).astype(np.float64)), (1, rep))
        if xi is only:
            assert np.abs(got[0].astype(np.float64) - ref[0]).max() <= 2.0 ** -126
            continue
        for i in range(mtok):
            e = exp if i == 1 else 0
            chk = check_against_oracle((got[i: i + 1] * 2.0 ** -e).astype(np.float32), (ref[i: i + 1] * 2.0 ** -e).astype(np.float32))
            assert chk.ok() and chk.within, (fmt, mtok, high, i, chk)


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
@pytest.mark.parametrize("big", [False, True])
@pytest.mark.parametrize("norm", [False, True])
def test_gemv_two_tokens(torch_gpu, fmt, big, norm, rng):
    """Two tokens on either side of the weight bytes where gemv_rowm takes over (20 MiB, FP8 40): the plan, the rows against the
    oracle's float64 product, with a workspace too small for any scratch as well (a plan without splits takes none)."""
    import ctypes as C
    from monolith_mi355 import kernels
    from monolith_mi355.runtime import hip
    torch = torch_gpu
    from monolith_mi355.formats.pack import two_tokens_on_matrix_cores
    k = 3072
    per_row = {"nvfp4": 1728, "int4_affine": 1728, "fp8_e4m3": 3072, "bf16": 6144}[fmt]
    n = (((40 if fmt == "fp8_e4m3" else 20) << 20) // (per_row * 16) + (1 if big else -1)) * 16
    assert two_tokens_on_matrix_cores(fmt, n, k) == big
    block = _matrix(fmt, 512, k, rng)                       # 512 random rows down the matrix
    rep = -(-n // 512)
    m = {kk: (np.tile(v, (rep, 1))[:n].copy() if isinstance(v, np.ndarray) and v.ndim == 2 else v) for kk, v in block.items()}
    x = rbf(rng.standard_normal((2, k)).astype(np.float32))
    nw = (1.0 + rng.standard_normal(k) * 0.1).astype(np.float32)
    w, xd = _upload(torch, m), to_dev_bf16(torch, x)
    kw = dict(norm_w=torch.from_numpy(nw).cuda(), eps=1e-6) if norm else {}
    d, _ = kernels._gemv_desc(w, xd, out_f32=True, **kw)
    plan = (C.c_int32 * 7)()
    hip.call("mi_gemv_plan", C.byref(d), plan)
    assert plan[0] == (3 if big else 1)
    xin = rbf(x / np.sqrt((x.astype(np.float64) ** 2).mean(-1, keepdims=True) + 1e-6) * nw) if norm else x
    ref = ON.matmul_acc(xin, _dequant(block))
    ref = np.tile(ref, (1, rep))[:, :n]
    small = torch.zeros(1024, dtype=torch.uint8, device="cuda")
    for ws in (None,) if fmt == "bf16" else (None, small):   # BF16 at this K splits on gemv_row too: it needs partials
        got = kernels.gemv(w, xd, out_f32=True, workspace=ws, **kw).cpu().numpy()
        chk = check_against_oracle(got, ref)
        assert (chk.ok_rounded() if norm else chk.ok()) and chk.within, (fmt, big, norm, chk)


@pytest.mark.parametrize("fmt,n,k", [("nvfp4", 12296, 3200), ("nvfp4", 7000, 6144), ("int4_affine", 12296, 3200),
                                     ("fp8_e4m3", 13720, 3136), ("fp8_e4m3", 170056, 3072), ("bf16", 5320, 2080)])
def test_gemv_two_tokens_norm_in_one_launch(torch_gpu, fmt, n, k, monkeypatch):
    """Two tokens on gemv_rowm with the input norm fused, over a last slice of one chunk, whole slices up to twelve
    waves, and more tiles than one round of workgroups: the bits of norm_apply and the plain GEMV after it (at a row
    stride past K), of mi_gemv_noalloc, and of a graph captured before any eager call on its stream, replayed with
    eager work between; the plain GEMV's rows against the decoded matrix in float64. The packed bytes are random."""
    import ctypes as C
    from monolith_mi355 import kernels
    from monolith_mi355.formats.pack import pack_bytes
    from monolith_mi355.runtime import hip
    torch = torch_gpu
    g = torch.Generator(device="cuda")
    g.manual_seed(n + k)
    data = torch.randint(0, 256, (pack_bytes(fmt, n, k),), dtype=torch.uint8, generator=g, device="cuda")
    data &= {"fp8_e4m3": 0xF7, "bf16": 0xBF}.get(fmt, 0x3F)      # finite codes, BF16 weights and scales
    rs = torch.rand((n + 15) // 16 * 16, generator=g, device="cuda") if fmt in ("nvfp4", "fp8_e4m3") else None
    w = kernels.PackedWeight(fmt, n, k, 1, data, rs)
    x = torch.randn(2, k + 24, generator=g, device="cuda").to(torch.bfloat16)[:, :k]
    nw = 1.0 + 0.1 * torch.randn(k, generator=g, device="cuda")
    kw = dict(norm_w=nw, eps=1e-6, out_f32=True)
    assert _plan(w, x, **kw)[0] == 3
    xn = kernels.norm_apply(x, nw, eps=1e-6)
    want = kernels.gemv(w, xn, out_f32=True)
    wd = kernels.dequant(w)
    for lo in range(0, n, 32768):
        part = wd[lo: lo + 32768].double()
        bound = xn.double().abs() @ part.abs().T                 # 32-bit sums of k products: a part of sum |x·w|
        assert ((want[:, lo: lo + 32768].double() - xn.double() @ part.T).abs() <= 2.0 ** -18 * bound).all()
    assert torch.equal(kernels.gemv(w, x, **kw), want)
    for rt in (1, 2, 3, 4, 5, 7):                                 # every tail of the tile loops
        monkeypatch.setenv("MI_GEMV_ROWM", f"0,{rt}")
        launch = _plan(w, x, **kw)
        assert launch[0] == 3 and launch[3] == rt, launch
        assert torch.equal(kernels.gemv(w, x, **kw), want), rt
    monkeypatch.delenv("MI_GEMV_ROWM")
    out = torch.zeros_like(want)
    d, _ = kernels._gemv_desc(w, x, out=out, **kw)
    torch.cuda.synchronize()
    hip.call("mi_gemv_noalloc", C.byref(d), hip.stream_handle())
    assert torch.equal(out, want)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = hip.Graph(s)
    with torch.cuda.stream(s), graph:
        kernels.gemv(w, x, out=out, **kw)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        graph.launch()
        s.synchronize()
        assert torch.equal(out, want)


def test_fp8_dequant_every_code(torch_gpu):
    """Every finite E4M3 code (signed zero, subnormals, ±448) decodes bit-exactly; the tensor scale multiplies once."""
    from monolith_mi355 import kernels
    from oracle.fp import e4m3_to_f32
    codes = np.array([c for c in range(256) if c & 0x7F != 0x7F], np.uint8)
    w = np.resize(codes, (32, 256)).astype(np.uint8)
    for s in (1.0, 0.0123):
        m = {"format": "fp8_e4m3", "weight": w, "weight_scale": float(np.float32(s))}
        got = kernels.dequant(_upload(torch_gpu, m)).cpu().numpy()
        ref = (e4m3_to_f32(w) * np.float32(s)).astype(np.float32)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), s


def test_gemv_split_k_fold_in_kernel(torch_gpu):
    """Split-K plans of gemv_row (M ≤ 2) fold their splits inside the kernel (gemv_rowm, M ≥ 3, in the reduction
    launch, which measured faster there) (arrival counters in the workspace): shapes with
    different tile counts interleaved, each repeated — the counters re-arm, the partials of one shape never disturb
    another's, the results repeat bit for bit, match the oracle, and a caller's zeroed workspace gives the same bits."""
    torch = torch_gpu
    import ctypes as C
    from monolith_mi355 import kernels
    from monolith_mi355.runtime import hip
    rng = np.random.default_rng(77)
    cases = []
    for n, k, mtok in [(4096, 12288, 1), (5120, 17408, 1), (1040, 17408, 2), (5120, 12288, 2), (5120, 17408, 8),
                       (2048, 17408, 5)]:
        m = _matrix("nvfp4", n, k, rng)
        w = _upload(torch, m)
        x = rbf(rng.standard_normal((mtok, k)))
        xd = to_dev_bf16(torch, x)
        yd = torch.empty(mtok, n, dtype=torch.float32, device="cuda")
        d = hip.MiGemvDesc(format=1, n=n, k=k, m=mtok, w=hip.ptr(w.data), row_scale=hip.ptr(w.row_scale),
                           x=hip.ptr(xd), ldx=k, y=hip.ptr(yd), ldy=n, out_f32=1)
        plan = (C.c_int32 * 7)()
        hip.call("mi_gemv_plan", C.byref(d), plan)
        assert plan[0] in (1, 3) and plan[4] > 1, (n, k, list(plan))     # gemv_row / gemv_rowm with K splits
        cases.append((m, w, x, xd, d))
    first = []
    for rep in range(3):
        for i, (m, w, x, xd, d) in enumerate(cases):
            y = kernels.gemv(w, xd, out_f32=True)
            torch.cuda.synchronize()
            y = y.cpu().numpy()
            if rep == 0:
                chk = check_against_oracle(y, ON.matmul_acc(x, _dequant(m)))
                assert chk.ok() and chk.within, (i, chk)
                first.append(y)
            else:
                assert np.array_equal(y, first[i]), (rep, i)
    ws_bytes = max(hip.load().mi_gemv_workspace_bytes(C.byref(d)) for *_, d in cases)
    ws = torch.zeros(ws_bytes, dtype=torch.uint8, device="cuda")
    for i, (m, w, x, xd, d) in enumerate(cases * 2):
        y = kernels.gemv(w, xd, out_f32=True, workspace=ws)
        torch.cuda.synchronize()
        assert np.array_equal(y.cpu().numpy(), first[i % len(cases)]), i


@pytest.mark.parametrize("fmt,n,k,mtok,epi,env", [
    ("nvfp4", 5120, 17408, 8, "residual", {}),              # gemv_rowm, K splits: the reduction writes x_next
    ("nvfp4", 5120, 17408, 3, "residual", {}),
    ("int4_affine", 2048, 8192, 8, "residual", {}),
    ("nvfp4", 1040, 17408, 1, "residual", {"MI_GEMV_FOLD": "0"}),   # gemv_row splits through the reduction launch
    ("nvfp4", 5120, 17408, 1, "residual", {}),              # splits folded in the kernel: a norm launch follows
    ("nvfp4", 2048, 5120, 8, None, {}),                     # one split: a norm launch follows
    ("nvfp4", 3000, 12288, 8, None, {}),                    # ragged N (whole 8-column vectors)
    ("nvfp4", 8192, 12288, 4, "residual", {}),              # the widest row one reduction workgroup takes
    ("nvfp4", 8200, 12288, 4, "residual", {}),              # wider: the reduction, then a norm launch
    ("nvfp4", 1032, 12288, 16, "residual", {}),             # N not a multiple of 16, sixteen tokens
    ("fp8_e4m3", 5120, 17408, 8, "residual", {}),           # per-row scales applied in the reduction
    ("bf16", 2048, 8192, 8, None, {}),                      # BF16 weights
])
def test_gemv_next_norm(torch_gpu, fmt, n, k, mtok, epi, env, rng, monkeypatch):
    """``next_norm``: y is bit-identical to the same GEMV without it, and x_next bit-identical to ``norm_apply`` of
    that y (the next GEMV's M ≥ 3 input norm), whichever launch computes it."""
    torch = torch_gpu
    from monolith_mi355 import kernels
    for kk, v in env.items():
        monkeypatch.setenv(kk, v)
    m = _matrix(fmt, n, k, rng)
    w = _upload(torch, m)
    xd = to_dev_bf16(torch, rbf(rng.standard_normal((mtok, k))))
    res = to_dev_bf16(torch, rbf(rng.standard_normal((mtok, n + 24))))[:, :n] if epi else None   # row stride > n
    nw = torch.from_numpy((1.0 + rng.standard_normal(n) * 0.1).astype(np.float32)).cuda()
    y0 = kernels.gemv(w, xd, epilogue=epi, residual=res)
    x0 = kernels.norm_apply(y0, nw, eps=1e-6)
    xn = torch.full((mtok, n), 7.0, dtype=torch.bfloat16, device="cuda")
    for rep in range(2):
        y1 = kernels.gemv(w, xd, epilogue=epi, residual=res, next_norm=(nw, xn, 1e-6))
        torch.cuda.synchronize()
        assert torch.equal(y1.view(torch.int16), y0.view(torch.int16)), rep
        assert torch.equal(xn.view(torch.int16), x0.view(torch.int16)), rep
        xn.fill_(7.0)
