"""The C ABI without a GPU: the built ``libmi355.so`` loads and exports every entry point ``include/*.h`` declares;
host-only entry points (pack sizes, launch plans, argument validation) behave; the ctypes signature table covers
the header."""

import ctypes as C
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared():
    names = set()
    for h in (ROOT / "include").glob("*.h"):
        text = re.sub(r"/\*.*?\*/", "", h.read_text(), flags=re.S)
        names |= set(re.findall(r"\b(mi_[a-z0-9_]+)\s*\(", text))
    return names


def test_header_declares_entry_points():
    names = declared()
    assert {"mi_gemv", "mi_dequant", "mi_malloc", "mi_graph_launch"} <= names


def test_wrapper_names_a_wrong_operand():
    """An array that is no bfloat16 tensor (a NumPy one has no ``stride()``), or one of another shape or layout, is refused
    with the operand's name, whatever its type offers."""
    import numpy as np
    import torch

    from monolith_mi355 import kernels
    w = kernels.PackedWeight("bf16", 16, 64, 1, torch.zeros(16), None)
    bf = torch.zeros((2, 64), dtype=torch.bfloat16)
    for x in (np.zeros((2, 64), np.float32), bf.float(), bf[0], bf.T, torch.zeros((2, 64)).to_sparse()):
        with pytest.raises(ValueError, match="gemv x"):
            kernels.gemv(w, x)


def test_library_exports_every_declared_symbol():
    from monolith_mi355.runtime import hip
    lib = hip.load()
    missing = [n for n in sorted(declared()) if not hasattr(lib, n)]
    assert not missing, missing


def test_ctypes_table_covers_header():
    from monolith_mi355.runtime import hip
    assert declared() == set(hip.SIGNATURES), declared() ^ set(hip.SIGNATURES)


def test_pack_bytes_matches_host_pack():
    from monolith_mi355.formats import pack as P
    from monolith_mi355.runtime import hip
    lib = hip.load()
    for fmt, fid in hip.MI_FMT.items():
        for n, k in ((37, 512), (17408, 5120), (5120, 17408)):
            assert lib.mi_pack_bytes(fid, n, k) == P.pack_bytes(fmt, n, k)
    assert lib.mi_pack_bytes(1, 16, 100) == 0            # K not a multiple of the chunk


def _desc(hip, **kw):
    base = dict(format=1, n=17408, k=5120, m=1, w=256, x=256, ldx=5120, y=256, ldy=17408)
    base.update(kw)
    return hip.MiGemvDesc(**base)


@pytest.mark.parametrize("n,k,m", [(34816, 5120, 1), (5120, 17408, 1), (34816, 5120, 8), (5120, 17408, 8),
                                   (4096, 4096, 1), (1024, 2048, 16), (16, 128, 3), (5120, 17408, 2)])
def test_gemv_plans_fit_the_hardware(n, k, m):
    from monolith_mi355.runtime import hip
    out = (C.c_int32 * 7)()
    hip.call("mi_gemv_plan", C.byref(_desc(hip, n=n, k=k, m=m, ldx=k, ldy=n)), out)
    kernel, waves, kw, tb, ks, lds, wgs = list(out)
    chunks = k // 128
    # gemv_row (VALU) for M <= 2; gemv_rowm (MFMA) above from one slice of K (4 chunks) on, else gemv_tk
    assert kernel == (1 if m <= 2 else 3 if chunks % 4 == 0 else 2)
    assert 1 <= waves <= 16 and kw >= 1 and lds <= 160 * 1024 and wgs >= 1 and ks >= 1 and tb >= 1
    if kernel == 1:                                      # K splits of ≤ waves·kw chunks each
        assert kw in (4, 8, 16) and waves * kw * ks >= chunks
    elif kernel == 3:                                    # 4 chunks per wave, ≤ 12 waves per K split
        assert waves * 4 == kw and waves <= 12 and ks * kw >= chunks and (ks - 1) * kw < chunks
        assert tb * wgs >= -(-n // 16) * ks              # tiles per workgroup × workgroups cover every tile
    else:
        assert ks * kw >= chunks and (ks - 1) * kw < chunks
    ws = hip.load().mi_gemv_workspace_bytes(C.byref(_desc(hip, n=n, k=k, m=m, ldx=k, ldy=n)))
    assert (ws > 0) == (ks > 1)


@pytest.mark.parametrize("fmt,k", [("fp8_e4m3", 64), ("fp8_e4m3", 1536), ("fp8_e4m3", 2048), ("fp8_e4m3", 2560),
                                   ("fp8_e4m3", 3072), ("fp8_e4m3", 5120), ("fp8_e4m3", 17408), ("nvfp4", 512),
                                   ("nvfp4", 2048), ("nvfp4", 2560), ("nvfp4", 3072), ("nvfp4", 6144)])
def test_gemv_rowm_plans_cover_any_height(fmt, k):
    """gemv_rowm has a plan for every row count (a vocabulary-sized head among them), whose workgroups cover every tile
    with partials that fit LDS: FP8 has no other kernel at M >= 3."""
    from monolith_mi355.runtime import hip
    out = (C.c_int32 * 7)()
    for m in (3, 8, 16):
        for n in (16, 4096, 34816, 111000, 128256, 131072, 135000, 151936, 168000, 201088, 248320, 262144, 1 << 20):
            hip.call("mi_gemv_plan", C.byref(_desc(hip, format=hip.MI_FMT[fmt], n=n, k=k, m=m, ldx=k, ldy=n)), out)
            kernel, waves, kw, rt, ks, lds, wgs = list(out)
            assert kernel == 3 and lds <= 160 * 1024 and waves <= 12, (m, n, list(out))
            assert rt * (wgs // ks) >= -(-n // 16) and wgs % ks == 0, (m, n, list(out))


@pytest.mark.parametrize("fmt", ["nvfp4", "int4_affine", "fp8_e4m3", "bf16"])
def test_two_tokens_with_a_norm_take_no_scratch(fmt):
    """One token or two with a fused input norm are one launch without scratch, on either kernel: calls that overlap
    (graphs captured on one stream, threads that share one) have nothing in common to write."""
    from monolith_mi355.runtime import hip
    out, kernels = (C.c_int32 * 7)(), set()
    for n, k in ((512, 2048), (16480, 5120), (34816, 5120), (12288, 3072), (20480, 6144), (248320, 5120)):
        for m in (1, 2):
            d = _desc(hip, format=hip.MI_FMT[fmt], n=n, k=k, m=m, ldx=k, ldy=n, norm_w=256)
            hip.call("mi_gemv_plan", C.byref(d), out)
            if out[4] > 1:                                   # K splits (a long K): partials, with or without a norm
                d.norm_w = 0
                hip.call("mi_gemv_plan", C.byref(d), out)
                assert out[4] > 1, (n, k, m)
                continue
            kernels.add((m, out[0]))
            assert hip.load().mi_gemv_workspace_bytes(C.byref(d)) == 0, (n, k, m)
    assert {(1, 1), (2, 1), (2, 3)} <= kernels


@pytest.mark.parametrize("fmt,n,k,ms", [("bf16", 34816, 6656, (3, 4)), ("bf16", 34816, 8192, (3, 4)),
                                        ("bf16", 65536, 12288, (3,)), ("nvfp4", 262144, 8192, (3, 4)),
                                        ("nvfp4", 151936, 6656, (3,))])
def test_wide_matrices_of_long_k_take_no_scratch(fmt, n, k, ms):
    """Where gemv_tk streams a long K unsplit it stays: no partials, so a workspace of any size and a stream captured
    before its first eager call will do."""
    from monolith_mi355.runtime import hip
    out = (C.c_int32 * 7)()
    for m in ms:
        d = _desc(hip, format=hip.MI_FMT[fmt], n=n, k=k, m=m, ldx=k, ldy=n)
        hip.call("mi_gemv_plan", C.byref(d), out)
        assert out[0] == 2 and out[4] == 1 and hip.load().mi_gemv_workspace_bytes(C.byref(d)) == 0, (m, list(out))


@pytest.mark.parametrize("fmt,n,k,m,kernel", [
    ("int4_affine", 131072, 1664, 3, 2), ("int4_affine", 65536, 512, 16, 2), ("int4_affine", 248320, 256, 3, 2),
    ("int4_affine", 131072, 1024, 4, 3), ("int4_affine", 131072, 1664, 16, 3), ("int4_affine", 34816, 2048, 16, 3),
    ("int4_affine", 50176, 4096, 16, 3), ("int4_affine", 22528, 256, 10, 2), ("int4_affine", 22528, 256, 8, 3),
    ("bf16", 50720, 128, 3, 2), ("bf16", 50720, 512, 16, 2), ("bf16", 50720, 512, 8, 3),
    ("bf16", 131072, 1536, 16, 2), ("bf16", 131072, 1536, 8, 3), ("bf16", 248320, 1536, 3, 2), ("bf16", 34816, 2048, 16, 3),
    ("bf16", 89472, 256, 16, 2), ("nvfp4", 131072, 640, 16, 2), ("nvfp4", 131072, 640, 8, 3), ("nvfp4", 131072, 512, 16, 3),
    ("nvfp4", 248320, 1152, 5, 2), ("nvfp4", 201088, 640, 16, 3), ("fp8_e4m3", 131072, 640, 16, 3),
    ("bf16", 384, 2048, 16, 1), ("bf16", 257, 2048, 16, 3), ("bf16", 1792, 1024, 8, 3), ("bf16", 14336, 128, 5, 1),
    ("bf16", 64, 2048, 8, 1)])
def test_tall_and_small_matrices_keep_their_kernels(fmt, n, k, m, kernel):
    """At M >= 3 a tall matrix of a short K stays on gemv_tk where that streams it unsplit on full CUs, and a small BF16
    matrix in gemv_row's token passes where a tile's passes share an XCD's L2: either side of each line. Neither needs
    scratch."""
    from monolith_mi355.runtime import hip
    out = (C.c_int32 * 7)()
    d = _desc(hip, format=hip.MI_FMT[fmt], n=n, k=k, m=m, ldx=k, ldy=n)
    hip.call("mi_gemv_plan", C.byref(d), out)
    assert out[0] == kernel and out[4] == 1 and hip.load().mi_gemv_workspace_bytes(C.byref(d)) == 0, list(out)


def test_gemv_rejects_bad_descriptors_before_launch():
    from monolith_mi355.runtime import hip
    lib = hip.load()
    bad = [dict(format=9), dict(k=100), dict(m=0), dict(m=17), dict(ldx=64), dict(w=0), dict(x=8),
           dict(epilogue=1, residual=0), dict(epilogue=2, n=40, ldy=20), dict(ldy=16)]
    for kw in bad:
        assert lib.mi_gemv(C.byref(_desc(hip, **kw)), None) == 1, kw      # MI_E_INVALID, nothing enqueued
        assert hip.last_error().startswith("mi_gemv")


def test_ctypes_descriptors_match_the_header_layout(tmp_path):
    """Every ctypes mirror of a header struct has the C layout: each field's offset and the struct's size, from a
    small program compiled against ``include/lithos_mi355.h`` (a descriptor shorter than the C struct would let the
    library read past it)."""
    import shutil
    import subprocess
    from monolith_mi355.runtime import hip
    cc = shutil.which("gcc") or shutil.which("cc")
    if cc is None:
        pytest.skip("no C compiler")
    classes = [v for k, v in vars(hip).items()
               if isinstance(v, type) and issubclass(v, C.Structure) and k.startswith("Mi")]
    assert len(classes) >= 15

    def c_name(cls):
        return "mi" + re.sub(r"([A-Z])", lambda m: "_" + m.group(1).lower(), cls.__name__[2:])

    lines = ['#include <stdio.h>', '#include <stddef.h>', f'#include "{ROOT / "include" / "lithos_mi355.h"}"',
             "int main(void) {"]
    for cls in classes:
        n = c_name(cls)
        lines.append(f'  printf("{cls.__name__} size %zu\\n", sizeof({n}));')
        for f, _ in cls._fields_:
            lines.append(f'  printf("{cls.__name__} {f} %zu\\n", offsetof({n}, {f}));')
    lines.append("  return 0;\n}")
    src = tmp_path / "layout.c"
    src.write_text("\n".join(lines))
    exe = tmp_path / "layout"
    subprocess.run([cc, "-I", str(ROOT / "include"), str(src), "-o", str(exe)], check=True, capture_output=True)
    want = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        cls_name, field, value = line.split()
        want[(cls_name, field)] = int(value)
    for cls in classes:
        assert C.sizeof(cls) == want[(cls.__name__, "size")], (cls.__name__, C.sizeof(cls))
        for f, _ in cls._fields_:
            assert getattr(cls, f).offset == want[(cls.__name__, f)], (cls.__name__, f)
