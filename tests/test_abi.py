"""The C-ABI library loads without a GPU and exports every symbol the header declares;
argument checking and the launch-geometry query run on the host alone."""
import ctypes
import json
import os
import re

import pytest

from accera_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _declared(header="accera_mi355x_gemm.h"):
    text = open(os.path.join(ROOT, "include", header)).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(acc950_\w+)\s*\(", text)))


def test_every_declared_symbol_is_exported():
    names = _declared()
    assert len(names) >= 9 and set(_lib.EXPORTS) == set(names)
    L = ctypes.CDLL(_lib.LIB_PATH)
    for n in names:
        assert getattr(L, n) is not None, n
    # the measurement aids are a library of their own; the product library holds none of them
    probes = _declared("accera_mi355x_probes.h")
    assert set(_lib.PROBE_EXPORTS) == set(probes) and not set(probes) & set(names)
    P = ctypes.CDLL(_lib.PROBES_LIB_PATH)
    for n in probes:
        assert getattr(P, n) is not None, n
        assert not hasattr(L, n), f"{n} belongs in the probes library only"


def test_phase_probe_refuses_what_its_kernels_do_not_take_before_launching():
    """The timed kernels take whole 256x256 tiles of dense, aligned operands only; the probe says so itself and runs nothing
    (no GPU is needed to be refused)."""
    P = _lib.probes()
    out = (ctypes.c_double * 8)()
    ok_ptrs = (0x10000, 0x20000, 0x30000)
    for M, N, K in ((300, 512, 512), (512, 300, 512), (512, 512, 100), (128, 512, 512), (512, 512, 0)):
        rc = P.acc950_mfma_phase_probe(_lib.F16, _lib.F32, M, N, K, *ok_ptrs, out)
        assert rc == _lib.UNSUPPORTED and b"multiples of 256" in P.acc950_probes_last_error(), (M, N, K)
    assert P.acc950_mfma_phase_probe(_lib.I8, _lib.I32, 512, 512, 96, *ok_ptrs, out) == _lib.UNSUPPORTED          # K of 64 bytes
    assert P.acc950_mfma_phase_probe(_lib.F16, _lib.F32, 512, 512, 512, 0x10008, 0x20000, 0x30000, out) == _lib.UNSUPPORTED
    assert P.acc950_mfma_phase_probe(_lib.F32, _lib.F32, 512, 512, 512, *ok_ptrs, out) == _lib.UNSUPPORTED
    assert P.acc950_mfma_phase_probe(_lib.F16, _lib.I32, 512, 512, 512, *ok_ptrs, out) == _lib.INVALID_ARGUMENT
    assert P.acc950_mfma_phase_probe(_lib.F16, _lib.F32, 512, 512, 512, None, 0x20000, 0x30000, out) == _lib.INVALID_ARGUMENT
    with pytest.raises(_lib.Acc950Error) as e:
        _lib.mfma_phase_probe(_lib.F16, _lib.F32, 300, 512, 512, *ok_ptrs)
    assert e.value.code == _lib.UNSUPPORTED and "multiples of 256" in str(e.value)


def test_variant_table_is_described():
    assert _lib.num_variants() >= 8 and _lib.num_skinny_variants() >= 1
    names = [_lib.variant_name(v) for v in range(_lib.num_variants())]
    assert len(set(names)) == len(names)
    assert any("direct" in n for n in names) and any("edge" in n for n in names)
    assert "skinny" in _lib.variant_name(_lib.VARIANT_SKINNY_BASE)
    with pytest.raises(_lib.Acc950Error):
        _lib.variant_name(_lib.num_variants())


# launch geometry expectations for the BASELINE configurations: grid = tiles of the block
# tile, block = waves * 64 (Plan.py:937-956 derives the same quantities from the bound indices;
# mfma_tests.py:2562,2572 pins them as <<<dim3(...), dim3(...)>>> strings)
def test_launch_geometry_of_the_configs():
    g, b, lds, v = _lib.launch_geometry(_lib.F16, _lib.F32, 4096, 4096, 4096, (4096, 1), (4096, 1), (4096, 1))
    name = _lib.variant_name(v)
    bm, bn = map(int, re.search(r"mfma (\d+)x(\d+)", name).groups())
    assert g == [(4096 // bm) * (4096 // bn), 1, 1] and b[0] % 64 == 0 and lds == 2 * (bm + bn) * 128
    g, b, lds, v = _lib.launch_geometry(_lib.BF16, _lib.BF16, 4096, 3072, 768, (768, 1), (1, 768), (3072, 1))
    assert "B=col-major" in _lib.variant_name(v)
    g, b, lds, v = _lib.launch_geometry(_lib.I8, _lib.I32, 8192, 8192, 8192, (8192, 1), (8192, 1), (8192, 1))
    assert "mfma" in _lib.variant_name(v)
    g, b, lds, v = _lib.launch_geometry(_lib.F16, _lib.F16, 8, 11008, 4096, (4096, 1), (11008, 1), (11008, 1))
    assert "skinny" in _lib.variant_name(v) and g[0] * g[1] >= 43 and b[0] % 64 == 0
    g, b, lds, v = _lib.launch_geometry(_lib.F32, _lib.F32, 512, 512, 512, (512, 1), (512, 1), (512, 1))
    assert v == _lib.VARIANT_F32_MFMA and g[:2] == [16, 16]
    # sizes that are not multiples of the 16-byte vector take the MFMA kernel whose fill accepts unaligned chunks; an operand with
    # no unit stride falls to the thread-bound kernel; explicit variants refuse what they do not take
    g, b, lds, v = _lib.launch_geometry(_lib.F16, _lib.F32, 100, 71, 40, (40, 1), (71, 1), (71, 1))
    assert "any-alignment" in _lib.variant_name(v) and "mfma 64x64" in _lib.variant_name(v) and g == [4, 1, 1]
    g, b, lds, v = _lib.launch_geometry(_lib.F16, _lib.F32, 100, 71, 40, (80, 2), (71, 1), (71, 1))
    assert v == _lib.VARIANT_GENERIC and g[:2] == [2, 2]
    with pytest.raises(_lib.Acc950Error) as e:
        _lib.launch_geometry(_lib.F16, _lib.F32, 100, 71, 40, (40, 1), (71, 1), (71, 1), variant=0)
    assert e.value.code == _lib.UNSUPPORTED


def test_argument_checking_on_the_host():
    with pytest.raises(_lib.Acc950Error) as e:
        _lib.launch_geometry(_lib.I8, _lib.F32, 64, 64, 64, (64, 1), (64, 1), (64, 1))
    assert e.value.code == _lib.INVALID_ARGUMENT and "type pair" in str(e.value)
    with pytest.raises(_lib.Acc950Error):
        _lib.launch_geometry(_lib.F16, _lib.F32, -1, 64, 64, (64, 1), (64, 1), (64, 1))
    with pytest.raises(_lib.Acc950Error):
        _lib.launch_geometry(_lib.F16, _lib.F32, 64, 64, 64, (-64, 1), (64, 1), (64, 1))
    # null pointers are rejected before anything is launched
    rc = _lib.lib().acc950_gemm_relu(_lib.F16, _lib.F32, 64, 64, 64, None, 64, 1, None, 64, 1, None, 64, 1, 1, 1, None)
    assert rc == _lib.INVALID_ARGUMENT and b"null" in _lib.lib().acc950_last_error()
    # empty problems are a no-op
    assert _lib.lib().acc950_gemm_relu(_lib.F16, _lib.F32, 0, 64, 64, None, 64, 1, None, 64, 1, None, 64, 1, 1, 1, None) == 0


def test_sweep_tool_lists_the_variants_that_take_a_problem():
    """accera_amd.tune enumerates the points of the variant space for a shape (counterpart of
    get_variants, tools/benchmarkers/accera_gemm.py:187-348) without touching the GPU."""
    from accera_amd import tune
    c = tune.candidates(_lib.F16, _lib.F32, 4096, 4096, 4096, (4096, 1), (4096, 1), (4096, 1))
    names = [_lib.variant_name(v) for v, _ in c]
    assert any("pingpong" in n for n in names) and any("generic" in n for n in names)
    assert not any("skinny" in n or "A=col-major" in n or " B=col-major" in n for n in names)
    c = tune.candidates(_lib.F16, _lib.F16, 8, 11008, 4096, (4096, 1), (11008, 1), (11008, 1))
    assert any("skinny mfma" in _lib.variant_name(v) and sp == 4 for v, sp in c)
    c = tune.candidates(_lib.F16, _lib.F32, 1024, 1024, 1024, (1, 1024), (1024, 1), (1024, 1))
    assert all("A=col-major" in _lib.variant_name(v) or "generic" in _lib.variant_name(v) for v, _ in c)
    import csv, os
    with open(os.path.join(os.path.dirname(tune.__file__), "shapes", "transformer_gemm.csv")) as f:
        rows = list(csv.DictReader(f))
    assert len(rows) >= 10 and {"m", "n", "k", "transA", "transB", "alpha", "beta"} <= set(rows[0])


def test_sweep_tool_audits_the_library_s_own_choice(tmp_path):
    """accera_amd.tune --audit: the kernel and K slices the library takes by itself against the fastest row of a sweep csv."""
    import csv
    from accera_amd import tune
    v, ks = tune.own_choice(_lib.F16, _lib.F32, 4096, 4096, 4096, False, False, 1.0, 0.0)
    chosen = _lib.variant_name(v)
    assert "hand-laid loop" in chosen and ks == 1
    other = next(_lib.variant_name(i) for i in range(_lib.num_variants()) if "pingpong" in _lib.variant_name(i))
    rows = [dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=v, k_splits=0, kernel=chosen, time_ms=0.1),
            dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=0, k_splits=0, kernel=other, time_ms=0.08),
            dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f16", variant=-2, k_splits=0, kernel="vendor library (torch.matmul)", time_ms=0.01)]
    path = tmp_path / "sweep.csv"
    with open(path, "w", newline="") as f:
        w = csv.DictWriter(f, fieldnames=list(rows[0]))
        w.writeheader()
        w.writerows(rows)
    lines = []
    geomean, worst = tune.audit(str(path), log=lines.append)
    assert abs(geomean - 1.25) < 1e-9 and len(worst) == 1 and worst[0][2] == chosen and worst[0][5] == other   # (the vendor row is no candidate)
    assert "1 problems" in lines[-1] and "1.2500" in lines[-1]


def test_choices_of_the_cost_model():
    """What the library takes by itself where measurements decided it (numbers in capi.hip next to each rule)."""
    from accera_amd import tune
    name = lambda *a: (lambda v, ks: (_lib.variant_name(v), ks))(*tune.own_choice(*a))
    # a last round that is half empty does not cost a whole round: one and a half rounds of 256 x 256 tiles stay on the four-wave kernel
    n, ks = name(_lib.F16, _lib.F16, 2048, 12288, 4096, False, False, 1.0, 0.0)
    assert "256x256" in n and "hand-laid loop" in n and ks == 1
    # a short K is not split, however few the tiles; a long one is
    assert name(_lib.F16, _lib.F16, 256, 256, 256, False, False, 1.0, 1.0)[1] == 1
    assert name(_lib.F16, _lib.F16, 64, 1152, 448, False, False, 1.0, 0.0)[1] == 1
    assert name(_lib.F16, _lib.F16, 2048, 256, 1536, False, False, 1.0, 0.0)[1] == 1      # (128 tiles: the partial sums cost more than the slices save)
    assert name(_lib.F16, _lib.F16, 64, 320, 1728, False, False, 1.0, 0.0)[1] > 1
    assert name(_lib.F16, _lib.F16, 768, 320, 30522, False, False, 1.0, 0.0)[1] >= 8
    # register-staged kernels (unaligned K): their steps are worth three of the direct kernels', no more
    assert name(_lib.F16, _lib.F16, 512, 128, 196, True, False, 1.0, 1.0)[1] == 1
    assert name(_lib.F16, _lib.F16, 6272, 32, 513, False, False, 1.0, 0.0)[1] == 1
    assert name(_lib.F16, _lib.F16, 196, 64, 801, False, False, 1.0, 0.0)[1] > 1
    # 128 x 128 tiles, two workgroups per CU: two stages of 128 bytes of K
    n, _ = name(_lib.F16, _lib.F16, 3072, 2304, 4096, False, True, 1.0, 1.0)
    assert ("128x128 kb128" in n and "stages=2" in n) or "256x256" in n
    # fp32: tiled kernels with direct fills where they apply, the kernel of 32 x 32 blocks for one round of blocks (512^3) and against the register-staged kernels
    assert "fp32 mfma 32x32" in name(_lib.F32, _lib.F32, 512, 512, 512, False, False, 1.0, 0.0)[0]
    assert "64x64" in name(_lib.F32, _lib.F32, 1152, 384, 64, True, False, 1.0, 1.0)[0]
    n, ks = name(_lib.F32, _lib.F32, 768, 576, 1024, False, False, 1.0, 1.0)
    assert "fill=direct" in n and ks > 1
    assert "fp32 mfma 32x32" in name(_lib.F32, _lib.F32, 800, 126, 49, True, False, 1.0, 1.0)[0]
    # few rows of A: the streaming kernel's 64-column blocks for the decode shape of the benchmark, its 256-column blocks (with
    # the K split that fills the chip in one round) once there are enough of them or the default would stream half lines
    narrow, wide = "skinny mfma cols/wg=64 waves=4 depth=4", "skinny mfma cols/wg=256 waves=4 depth=4"
    assert name(_lib.F16, _lib.F16, 8, 11008, 4096, False, False, 1.0, 0.0) == (narrow, 1)
    assert name(_lib.F16, _lib.F16, 8, 16384, 4096, False, False, 1.0, 0.0) == (narrow, 1)     # (two slices would fill half the chip)
    assert name(_lib.F16, _lib.F16, 8, 16384, 8192, False, False, 1.0, 0.0) == (wide, 4)
    assert name(_lib.BF16, _lib.BF16, 8, 22016, 8192, False, False, 1.0, 0.0) == (wide, 2)
    assert name(_lib.F16, _lib.F16, 8, 65536, 8192, False, False, 1.0, 0.0) == (wide, 1)
    assert name(_lib.F16, _lib.F16, 8, 66048, 4096, False, False, 1.0, 0.0) == (narrow, 1)     # (258 wide blocks: a second round for two of them)
    assert name(_lib.F16, _lib.F16, 32, 16384, 8192, False, False, 1.0, 0.0) == (narrow, 1)    # (more rows: the second trip costs more)
    assert name(_lib.F16, _lib.F16, 32, 16384, 16384, False, False, 1.0, 0.0) == (wide, 4)
    assert name(_lib.I8, _lib.I32, 8, 12288, 16384, False, False, 1.0, 0.0) == (wide, 4)
    assert name(_lib.I8, _lib.I32, 8, 8192, 8192, False, False, 1.0, 0.0) == (wide, 4)
    assert name(_lib.I8, _lib.I32, 8, 4096, 8192, False, False, 1.0, 0.0)[0] == narrow
    # a few dozen to a few hundred rows against a B far beyond the caches: a tile as tall as A (B is streamed once) and the K
    # slices that make about 256 workgroups (512 of the register-staged ones); the slices alone from 64 MB of B on
    n, ks = name(_lib.F16, _lib.F16, 128, 16384, 16384, False, False, 1.0, 0.0)
    assert "128x128" in n and "fill=direct" in n and ks == 2
    n, ks = name(_lib.F16, _lib.F16, 33, 8192, 28672, False, False, 1.0, 0.0)
    assert "64x64" in n and "fill=direct" in n and ks == 4                              # (fewer rows than the tile has: direct fills all the same)
    n, ks = name(_lib.F16, _lib.F16, 100, 8192, 28672, False, False, 1.0, 0.0)
    assert "128x128" in n and "fill=direct" in n and ks == 4
    n, ks = name(_lib.F16, _lib.F16, 100, 8192, 28672, True, False, 1.0, 0.0)           # (a column-major A: the register-staged edge form)
    assert "128x128" in n and "edge" in n and ks == 8
    n, ks = name(_lib.F16, _lib.F16, 8, 11008, 4096, False, True, 1.0, 0.0)            # a decode step against a K-contiguous B
    assert "64x64" in n and "fill=direct" in n and ks == 1
    n, ks = name(_lib.F16, _lib.F16, 8, 4096, 4096, False, True, 1.0, 0.0)             # (fewer than 64 rows: from 16 MB of B on)
    assert "64x64" in n and "fill=direct" in n and ks == 4
    assert "edge" in name(_lib.F16, _lib.F16, 8, 2048, 2048, False, True, 1.0, 0.0)[0]  # (8 MB of B: as before)
    assert name(_lib.F16, _lib.F16, 64, 8192, 2048, False, False, 1.0, 0.0)[1] == 1     # (64 rows and 32 MB: the general rule's slices)
    n, ks = name(_lib.BF16, _lib.BF16, 256, 28672, 8192, False, False, 1.0, 0.0)
    assert "256x256" in n and "hand-laid loop" in n and ks == 2
    n, ks = name(_lib.F16, _lib.F16, 256, 32000, 4096, False, False, 1.0, 0.0)
    assert "256x256" in n and ks == 1                                                    # (two slices' partial sums would be a quarter of B)
    n, ks = name(_lib.F16, _lib.F16, 64, 8192, 28672, False, True, 1.0, 0.0)
    assert "64x64" in n and "fill=direct" in n and ks == 4
    assert name(_lib.F16, _lib.F16, 64, 16384, 16384, False, False, 1.0, 0.0)[1] == 1   # (256 tiles stream by themselves)
    n, ks = name(_lib.F16, _lib.F16, 100, 11008, 4096, False, False, 1.0, 0.0)
    assert "64x64" in n and "fill=direct" in n and ks == 1                              # (90 MB: the general rule's tiles, 344 of them)


@pytest.mark.parametrize("M,N,K,tile,slices", [
    (31, 4416, 9792, "64x64", 7), (17, 4096, 4096, "64x64", 4), (32, 64, 262144, "64x64", 32), (24, 5056, 8192, "64x64", 6), (17, 6400, 3584, "64x64", 3),
    (31, 20800, 4544, "64x64", 1),          # (325 tiles: unsplit, they fill the chip)
    (31, 9600, 1792, None, 1), (24, 9600, 2048, None, 1), (17, 6400, 2624, None, 1),  # (two slices or none: the streaming kernel)
    (17, 6080, 3264, None, None), (17, 8960, 5632, None, None), (32, 8960, 5632, "64x64", 3), (17, 9984, 8192, None, None), (17, 9600, 3584, "64x64", 3),
    (18, 8192, 2048, None, None), (17, 8192, 8192, None, None), (32, 8192, 8192, "64x64", 4),   # (rows of B 16 KB apart)
    (29, 11712, 7168, None, None), (25, 37056, 6912, None, None), (17, 24576, 8192, None, None),
    (22, 5056, 1408, None, None),           # (a B of less than 32 MB)
])
def test_17_to_32_rows_against_a_large_b(M, N, K, tile, slices):
    """Tiles in slices or the streaming kernel, as measured; an fp32 result and int8 keep the streaming kernel, whose sums are shorter chains."""
    from accera_amd import tune
    for t in (_lib.F16, _lib.BF16):
        v, ks = tune.own_choice(t, t, M, N, K, False, False, 1.0, 0.0)
        name = _lib.variant_name(v)
        assert ("mfma 64x64" in name and "fill=direct" in name) if tile else "skinny" in name, name
        assert slices is None or ks == slices, (name, ks)
        assert "skinny" in _lib.variant_name(tune.own_choice(t, _lib.F32, M, N, K, False, False, 1.0, 0.0)[0])
    assert "skinny" in _lib.variant_name(tune.own_choice(_lib.I8, _lib.I32, M, N, K, False, False, 1.0, 0.0)[0])


def test_slices_of_the_streaming_kernels():
    """As many as pay, not as many as there are CUs for; an fp32 result keeps the many (its sums are shorter chains)."""
    from accera_amd import tune
    own = lambda *a: tune.own_choice(*a, False, False, 1.0, 0.0)
    narrow = next(_lib.VARIANT_SKINNY_BASE + i for i in range(_lib.num_skinny_variants()) if "mfma cols/wg=64" in _lib.variant_name(_lib.VARIANT_SKINNY_BASE + i))
    for (M, N, K), slices, many in [((22, 5056, 1408), 1, 4), ((18, 3904, 2752), 1, 5), ((28, 3144, 3904), 3, 6), ((16, 1088, 5440), 5, 16), ((26, 1752, 1984), 4, 7)]:
        assert own(_lib.F16, _lib.F16, M, N, K) == (narrow, slices)
        assert own(_lib.BF16, _lib.BF16, M, N, K) == (narrow, slices)
        assert own(_lib.F16, _lib.F32, M, N, K) == (narrow, many)
    assert own(_lib.I8, _lib.I32, 28, 4096, 6144)[1] in (3, 4)   # (17.9 us unsplit, 11.5 in four)
    assert own(_lib.I8, _lib.I32, 15, 5696, 1536) == (narrow, 1)
    # never more than a workgroup per CU, nor slices of less than 256 rows of B
    for N in (64, 512, 1984, 4096, 8128):
        for K in (256, 500 // 32 * 32, 4096, 32768):
            s = own(_lib.F16, _lib.F16, 8, N, K)[1]
            assert s == 1 or (s * -(-N // 64) <= 256 and K // s >= 256)


def test_slices_against_a_k_contiguous_b():
    """Any number of slices up to 16, powers of two from there on."""
    from accera_amd import tune
    for (M, N, K), slices in [((48, 768, 23744), 16), ((2, 1664, 23744), 16), ((63, 2048, 6144), 6), ((48, 2560, 16384), 12), ((68, 5376, 23552), 6), ((11, 6208, 3904), 4)]:
        v, ks = tune.own_choice(_lib.F16, _lib.F16, M, N, K, False, True, 1.0, 0.0)
        assert "fill=direct" in _lib.variant_name(v) and ks == slices, (M, N, K, ks)


def test_tiles_of_register_staged_problems_with_a_short_k():
    """64 x 64 or 128 x 128 tiles by a model of both (unaligned operands, K of 64 to 2048 bytes), what reads C among it."""
    from accera_amd import tune
    tile = lambda v: re.search(r"mfma (\d+x\d+)", _lib.variant_name(v)).group(1)
    F16, BF16, F32, I8, I32 = _lib.F16, _lib.BF16, _lib.F32, _lib.I8, _lib.I32
    for (t, o, M, N, K, ta, beta), want in [
            ((F16, F16, 704, 3136, 52, False, 0.0), "64x64"), ((F16, F16, 4936, 643, 112, False, 0.0), "64x64"),
            ((F16, F32, 5184, 3972, 73, False, 0.0), "128x128"), ((BF16, BF16, 793, 5760, 547, True, 0.0), "128x128"),
            ((F16, F16, 824, 4072, 888, False, 0.0), "128x128"), ((F16, F32, 600, 901, 100, False, 1.0), "64x64")]:
        v, ks = tune.own_choice(t, o, M, N, K, ta, False, 1.0, beta)
        assert "edge" in _lib.variant_name(v) and tile(v) == want and ks == 1, (M, N, K, _lib.variant_name(v), ks)


def test_fp32_problems_with_unaligned_operands_and_a_short_k():
    """More 32 x 32 blocks than two rounds: the 64 x 64 tiles, whose sums are four chains as well, never the 128 x 128 ones; fewer, or
    tiles that would be mostly empty: the kernel of blocks."""
    from accera_amd import tune
    own = lambda *a: _lib.variant_name(tune.own_choice(_lib.F32, _lib.F32, *a, 1.0, 0.0)[0])
    for a in [(4864, 2754, 648, False, False), (4148, 1439, 128, False, False), (1472, 674, 576, False, False), (5037, 376, 33, False, True), (700, 901, 766, True, True)]:
        assert "mfma 64x64" in own(*a) and "edge" in own(*a), (a, own(*a))
    for a in [(520, 793, 448, False, False), (512, 1024, 33, False, True), (20000, 24, 100, False, False), (300, 301, 301, False, False)]:
        assert "fp32 mfma 32x32" in own(*a), (a, own(*a))
    # a batch counts with all its blocks (grid: 64 x 64 tiles of one problem, or its 32 x 32 blocks)
    geom = lambda batch: _batched_geometry(batch, 80, 192, 301)
    assert geom(104) == (6, 104) and geom(8)[1] == 8 and geom(8)[0] != 6


def _batched_geometry(batch, M, N, K):
    L, h, v, ks, P = _lib.lib(), ctypes.c_int(-1), ctypes.c_int(), ctypes.c_int(), ctypes.c_void_p
    _lib.check(L.acc950_bind(_lib.F32, _lib.F32, batch, M, N, K, P(1 << 32), M * K, K, 1, P(2 << 32), K * N, N, 1, P(3 << 32), M * N, N, 1,
                             _lib.PROLOGUE_SET0, 0.0, _lib.EPILOGUE_NONE, 0.0, _lib.VARIANT_AUTO, 0, None, ctypes.byref(h)))
    try:
        _lib.check(L.acc950_bound_choice(h.value, ctypes.byref(v), ctypes.byref(ks)))
    finally:
        L.acc950_unbind(h.value)
    if v.value == _lib.VARIANT_F32_MFMA:
        return (-1, batch)
    return _lib.launch_geometry(_lib.F32, _lib.F32, M, N, K, (K, 1), (N, 1), (N, 1), v.value)[0][0], batch


def test_bound_call_handles_without_launching():
    """acc950_bind validates and chooses once; handles are reused after acc950_unbind; unknown handles
    are reported.  (No launch here: there is no GPU on the CPU test tier.)"""
    import ctypes
    L = _lib.lib()
    h = ctypes.c_int(-1)
    args = (_lib.F16, _lib.F32, 1, 256, 256, 256, 0x10000, 0, 256, 1, 0x20000, 0, 256, 1, 0x30000, 0, 256, 1,
            _lib.PROLOGUE_SET0, 0.0, _lib.EPILOGUE_RELU, 0.0, _lib.VARIANT_AUTO, 0, None)
    assert L.acc950_bind(*args, ctypes.byref(h)) == _lib.OK and h.value >= 0
    first = h.value
    v, ks = ctypes.c_int(-5), ctypes.c_int(-5)
    assert L.acc950_bound_choice(first, ctypes.byref(v), ctypes.byref(ks)) == _lib.OK
    assert "mfma" in _lib.variant_name(v.value) and ks.value >= 1
    assert L.acc950_unbind(first) == _lib.OK
    assert L.acc950_unbind(first) == _lib.INVALID_ARGUMENT and L.acc950_launch(first) == _lib.INVALID_ARGUMENT
    assert L.acc950_bound_choice(first, ctypes.byref(v), ctypes.byref(ks)) == _lib.INVALID_ARGUMENT
    assert L.acc950_bind(*args, ctypes.byref(h)) == _lib.OK and h.value == first   # slot reused
    assert L.acc950_unbind(first) == _lib.OK
    bad = list(args)
    bad[6] = 0   # null A
    assert L.acc950_bind(*bad, ctypes.byref(h)) == _lib.INVALID_ARGUMENT
    bad = list(args)
    bad[22] = 57 + 1000   # unknown variant
    assert L.acc950_bind(*bad, ctypes.byref(h)) == _lib.INVALID_ARGUMENT
    # A's stride between consecutive k and B's between consecutive columns travel as 32-bit kernel arguments
    for where in (9, 13):   # a_col_stride, b_col_stride
        bad = list(args)
        bad[where] = 1 << 31
        assert L.acc950_bind(*bad, ctypes.byref(h)) == _lib.UNSUPPORTED and b"2^31" in L.acc950_last_error()


def test_tuned_table_is_consulted_by_name_and_validated(tmp_path, monkeypatch):
    """accera_amd.tuned: entries name kernels by description; unknown kernels and kernels the library
    refuses for the problem are ignored."""
    from accera_amd import tuned
    path = tmp_path / "tuned.json"
    monkeypatch.setenv("ACCERA_AMD_TUNED", str(path))
    rows = [dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=1, k_splits=0,
                 kernel=_lib.variant_name(1), time_ms=0.2, TFlops=1.0, correct=True),
            dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=0, k_splits=0,
                 kernel=_lib.variant_name(0), time_ms=0.3, TFlops=1.0, correct=True),
            dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=5, k_splits=0,
                 kernel=_lib.variant_name(5), time_ms=0.1, TFlops=1.0, correct=False),          # failed its check: never recorded
            dict(m=1000, n=1000, k=1000, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=1, k_splits=0,
                 kernel=_lib.variant_name(1), time_ms=0.1, TFlops=1.0, correct=True),           # kernel cannot take this shape
            dict(m=512, n=512, k=512, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=1, k_splits=0,
                 kernel="a kernel this library does not have", time_ms=0.1, TFlops=1.0, correct=True),
            dict(m=4096, n=4096, k=4096, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f32", variant=-2, k_splits=0,
                 kernel="vendor library (torch.matmul)", time_ms=0.05, TFlops=1.0, correct="")]
    assert tuned.save(rows, str(path)) == 3
    tuned.reset()
    args = (_lib.F16, _lib.F32, 4096, 4096, 4096, (4096, 1), (4096, 1), (4096, 1))
    assert tuned.lookup(*args, True) == (1, 0)                 # fastest verified row
    assert tuned.lookup(*args, False) is None                  # other op class: not recorded
    assert tuned.lookup(*args, "acc") is None and tuned.lookup(*args, "lean") == (1, 0)
    assert tuned.ops_class(_lib.PROLOGUE_SET0, 0.0, _lib.EPILOGUE_RELU) == "lean"
    assert tuned.ops_class(_lib.PROLOGUE_NONE, 0.0, _lib.EPILOGUE_NONE) == "acc"
    assert tuned.ops_class(_lib.PROLOGUE_SET, 1.0, _lib.EPILOGUE_RELU) == "full"
    assert tuned.ops_class(_lib.PROLOGUE_NONE, 0.0, _lib.EPILOGUE_SCALE) == "full"
    assert tuned.lookup(_lib.F16, _lib.F32, 1000, 1000, 1000, (1000, 1), (1000, 1), (1000, 1), True) is None
    assert tuned.lookup(_lib.F16, _lib.F32, 512, 512, 512, (512, 1), (512, 1), (512, 1), True) is None
    assert tuned.lookup(_lib.F16, _lib.F32, 4096, 4096, 4096, (4096, 1), (4096, 1), (4100, 1), True) is None  # padded C: not a table shape
    tuned.reset()


def test_recorded_choices_without_asking_the_library(tmp_path, monkeypatch):
    """tuned.recorded, which an eager call uses, finds what tuned.lookup finds wherever the library takes the recorded kernel."""
    from accera_amd import tuned
    F, name = _lib.F16, _lib.variant_name(7)
    col = next(_lib.variant_name(v) for v in range(_lib.num_variants()) if "A=col-major" in _lib.variant_name(v) and "edge" in _lib.variant_name(v))
    path = tmp_path / "table.json"
    path.write_text(json.dumps({
        tuned.key(F, F, 256, 512, 128, False, False, "lean"): {"kernel": name, "k_splits": 1},
        tuned.key(F, F, 256, 512, 128, True, False, "acc"): {"kernel": col, "k_splits": 0},
        tuned.key(F, F, 1, 512, 128, False, False, "lean"): {"kernel": "no such kernel", "k_splits": 0},
        "not a key": {"kernel": name}}))
    monkeypatch.setenv("ACCERA_AMD_TUNED", str(path))
    tuned.reset()
    try:
        for M, a, c, ops in ((256, (128, 1), (512, 1), "lean"), (256, (1, 256), (512, 1), "acc"), (256, (1, 256), (512, 1), "lean"), (256, (136, 1), (512, 1), "lean"),
                             (256, (128, 1), (520, 1), "lean"), (1, (128, 1), (512, 1), "lean"), (257, (128, 1), (512, 1), "lean")):
            want = tuned.lookup(F, F, M, 512, 128, a, (512, 1), c, ops)
            assert tuned.recorded(F, F, M, 512, 128, *a, 512, 1, *c, ops) == want, (M, a, c, ops)
        assert tuned.recorded(F, F, 256, 512, 128, 128, 1, 512, 1, 512, 1, "lean") == (7, 1)
    finally:
        monkeypatch.undo()
        tuned.reset()


def test_a_recorded_short_k_kernel_is_found(tmp_path, monkeypatch):
    """What a sweep saves for the short-K kernel, which it tries like any other, is what the look-ups of both kinds of call find."""
    from accera_amd import tune, tuned
    M, N, K = 12544, 1024, 128
    assert (_lib.VARIANT_SHORT_K, 0) in tune.candidates(_lib.F16, _lib.F16, M, N, K, (K, 1), (N, 1), (N, 1))
    path = tmp_path / "table.json"
    row = dict(m=M, n=N, k=K, transA=0, transB=0, alpha=1.0, beta=0.0, type="f16", out_type="f16", variant=_lib.VARIANT_SHORT_K, k_splits=0,
               kernel=_lib.variant_name(_lib.VARIANT_SHORT_K), time_ms=0.01, TFlops=1.0, correct=True)
    monkeypatch.setenv("ACCERA_AMD_TUNED", str(path))
    assert tuned.save([row], str(path)) == 1
    tuned.reset()
    try:
        assert tuned.lookup(_lib.F16, _lib.F16, M, N, K, (K, 1), (N, 1), (N, 1), "lean") == (_lib.VARIANT_SHORT_K, 0)
        assert tuned.recorded(_lib.F16, _lib.F16, M, N, K, K, 1, N, 1, N, 1, "lean") == (_lib.VARIANT_SHORT_K, 0)
    finally:
        monkeypatch.undo()
        tuned.reset()


def test_packed_call_checks_its_numbers():
    import struct
    pack = struct.Struct("19qdqd3q").pack
    L = _lib.lib()
    head = [_lib.F16, _lib.F16, 1, 64, 64, 64] + [0, 0, 64, 1] * 3
    assert L.acc950_gemm_packed(None) == _lib.INVALID_ARGUMENT
    assert L.acc950_gemm_packed(pack(*head, 1, 0.0, 1, 0.0, -1, 0, 0)) == _lib.INVALID_ARGUMENT  # (null matrices)
    assert "null" in L.acc950_last_error().decode()
    for i in (0, 2, 3, 5):
        wide = list(head)
        wide[i] += 1 << 32
        assert L.acc950_gemm_packed(pack(*wide, 1, 0.0, 1, 0.0, -1, 0, 0)) == _lib.INVALID_ARGUMENT and "32-bit" in L.acc950_last_error().decode()
    empty = list(head)
    empty[3] = 0
    assert L.acc950_gemm_packed(pack(*empty, 1, 0.0, 1, 0.0, -1, 0, 0)) == _lib.OK  # (nothing to do)


@pytest.mark.parametrize("in_type,M,N,K,b_col,tile,slices", [
    ("f16", 127, 14784, 4096, True, "128x128", 2),     # 116 tiles: two slices of each
    ("bf16", 169, 6336, 6656, False, "128x128", 2),
    ("f16", 100, 12800, 4096, False, "64x64", 1),      # a row-major B, slices of 2048: the general rule's tiles
    ("bf16", 107, 6016, 3648, True, "64x64", 1),       # three slices' sums are more than a sixth of B, two are 94 workgroups
    ("i8", 155, 5568, 7296, False, "128x128", 2), ("i8", 92, 9920, 7936, True, "128x128", 3), ("i8", 194, 2304, 14720, False, "128x128", 4),
    ("i8", 100, 6080, 3456, True, "64x64", 1),         # a B of 20 MB
    ("i8", 181, 5440, 7616, True, "64x64", 1),         # K of no whole 128 bytes
    # no slices of these tiles: the general rule's, which read B as often and fill the chip
    ("f16", 121, 12800, 1536, True, "64x64", 1), ("bf16", 69, 14336, 1600, True, "64x64", 1), ("f16", 105, 13056, 1792, True, "64x64", 1), ("i8", 249, 7680, 5120, True, "64x64", 1),
    ("bf16", 245, 6720, 4672, True, "128x128", 2),     # (two slices by the general rule's count)
    ("f16", 86, 13312, 2240, True, "128x128", 2), ("f16", 77, 15360, 1984, True, "64x64", 1), ("i8", 70, 13312, 3200, True, "64x64", 1),  # a K-contiguous B: from a K of 2048, int8 3800
    ("i8", 66, 10752, 3840, True, "128x128", 3), ("i8", 105, 16320, 4096, True, "64x64", 1), ("i8", 105, 16320, 4352, True, "128x128", 2), ("i8", 127, 7936, 4864, True, "64x64", 1),  # ... by the number of smaller tiles
    ("i8", 246, 4992, 9920, False, "128x128", 3),      # the general rule's three slices of these tiles, not two
    ("i8", 124, 3584, 10112, True, "64x64", 4), ("i8", 124, 3584, 10112, False, "128x128", 5),
    ("i8", 144, 14581, 5122, True, "128x128", 1), ("i8", 191, 13089, 6526, False, "128x128", 1),   # register-staged tiles: the sums of two slices are too much beside B
    ("i8", 92, 16535, 4956, False, "128x128", 3), ("i8", 78, 21032, 5208, True, "128x128", 3),     # ... three pay for themselves
])
def test_65_to_256_rows_against_32_to_192_mb(in_type, M, N, K, b_col, tile, slices):
    from accera_amd import tune
    i, o = {"f16": (_lib.F16, _lib.F16), "bf16": (_lib.BF16, _lib.BF16), "i8": (_lib.I8, _lib.I32)}[in_type]
    variant, splits = tune.own_choice(i, o, M, N, K, False, b_col, 1.0, 0.0)
    assert f"mfma {tile} " in _lib.variant_name(variant) and splits == slices, (_lib.variant_name(variant), splits)


@pytest.mark.parametrize("in_type,M,N,K,slices", [("i8", 67, 10112, 3584, 3), ("i8", 105, 11520, 4096, 2), ("i8", 80, 3712, 9472, 7), ("bf16", 102, 12800, 2240, 1)])
def test_65_to_256_rows_against_a_k_contiguous_b_reading_c(in_type, M, N, K, slices):
    """The general rule's tiles are register-staged here: the 128 x 128 ones with direct fills, in slices or not."""
    from accera_amd import tune
    i, o = {"bf16": (_lib.BF16, _lib.BF16), "i8": (_lib.I8, _lib.I32)}[in_type]
    variant, splits = tune.own_choice(i, o, M, N, K, False, True, 1.0, 0.5)
    name = _lib.variant_name(variant)
    assert "mfma 128x128 " in name and "fill=direct" in name and splits == slices, (name, splits)


@pytest.mark.parametrize("in_type,M,N,K,tile,slices", [
    ("f16", 1234, 5678, 4321, "256x256", 2), ("f16", 3913, 893, 6825, "256x256", 4), ("bf16", 703, 3293, 5909, "256x256", 6), ("i8", 644, 7700, 5155, "256x256", 2),
    ("f16", 1234, 5678, 3333, "128x128", 1),      # K too short for the sums of the slices
    ("f16", 2600, 2900, 4321, "128x128", 1),      # 132 tiles: no two slices of each
    ("i8", 2576, 2645, 6001, "128x128", 1),
    ("f16", 520, 8001, 4321, "128x128", 1),       # a last row of tiles that is nearly empty
    ("i8", 5184, 736, 5790, "256x256", 4),
])
def test_large_tiles_in_slices_for_unaligned_problems_with_a_long_k(in_type, M, N, K, tile, slices):
    from accera_amd import tune
    i, o = {"f16": (_lib.F16, _lib.F16), "bf16": (_lib.BF16, _lib.BF16), "i8": (_lib.I8, _lib.I32)}[in_type]
    variant, splits = tune.own_choice(i, o, M, N, K, False, False, 1.0, 0.0)
    assert f"mfma {tile} " in _lib.variant_name(variant) and "any-alignment" in _lib.variant_name(variant) and splits == slices, (_lib.variant_name(variant), splits)


def _host_parts(tin, tout, M, N, K, a=1 << 40, b=2 << 40, c=3 << 40, a_rs=None, c_rs=None, b_strides=None, prologue=1, batch=1):
    import struct
    parts, (b_rs, b_cs) = ctypes.c_int(-1), b_strides or (N, 1)
    call = struct.Struct("19qdqd3q").pack(tin, tout, batch, M, N, K, a, M * K * (batch > 1), a_rs or K, 1, b, K * N * (batch > 1), b_rs, b_cs, c, M * N * (batch > 1), c_rs or N, 1,
                                          prologue, 0.0, _lib.EPILOGUE_RELU, 0.0, _lib.VARIANT_AUTO, 0, 0)
    _lib.check(_lib.lib().acc950_host_parts(call, ctypes.byref(parts)))
    return parts.value


def test_host_calls_whose_operands_overlap_go_in_one_piece():
    """In parts, C's first rows are written while A's later rows are unread: not where they are the same bytes."""
    F16, F32 = _lib.F16, _lib.F32
    n, row, x = 4096, 2 * 4096, 1 << 40
    whole = _host_parts(F16, F16, n, n, n)
    assert whole == 4
    assert _host_parts(F16, F16, n, n, n, a=x, c=x + row) == 1                       # A = X[:-1], C = X[1:]
    assert _host_parts(F16, F16, n, n, n, a=x, c=x + 2) == 1                         # one element on
    assert _host_parts(F16, F16, n, n, n, a=x, c=x + (n - 1) * row) == 1             # C over A's last row
    assert _host_parts(F16, F32, n, n, n, a=x, c=x) == 1                             # an fp16 A at the start of an fp32 C's buffer
    assert _host_parts(F16, F16, n, n, n, a=x, c=x, a_rs=n + 8) == whole             # C's rows lie before A's of the same number ...
    assert _host_parts(F16, F16, n, n, n, a=x + row, c=x) == whole                   # ... A = X[1:], C = X[:-1]
    assert _host_parts(F16, F16, n, n, n, a=x, c=x) == whole                         # the same array
    assert _host_parts(F16, F16, n, n, n, b=3 << 40) == whole                        # C over B, which is read first
    assert _host_parts(F16, F16, n, n, n, a=x, c=x + n * row) == whole               # neighbours
    assert _host_parts(F16, F16, n, n, n, prologue=0) == 1 and _host_parts(F16, F16, n, n, n, batch=2) == 1 and _host_parts(F16, F16, 0, n, n) == 0
    parts = ctypes.c_int()
    assert _lib.lib().acc950_host_parts(None, ctypes.byref(parts)) == _lib.INVALID_ARGUMENT


@pytest.mark.parametrize("tin,tout,M,N,K,parts", [
    ("f16", "f32", 4096, 4096, 4096, 8), ("f16", "f16", 2048, 2048, 2048, 4),
    ("f32", "f32", 4096, 4096, 4096, 2),      # eight parts: 16 of 256 CUs' worth of tiles each, 6674 us for 4239
    ("f32", "f32", 1500, 3000, 2000, 2), ("f32", "f32", 1024, 8192, 8192, 2),
    ("i8", "i32", 1024, 16384, 1024, 1),      # nothing of A to overlap with C
    ("i8", "i32", 1536, 3000, 333, 1), ("f16", "f16", 511, 16384, 256, 1), ("f16", "f32", 1024, 1024, 1024, 1),
])
def test_host_calls_go_in_as_many_parts_as_pay(tin, tout, M, N, K, parts):
    """Parts that leave the chip idle, or that have nothing to overlap, are not made."""
    ids = {"f16": _lib.F16, "f32": _lib.F32, "i8": _lib.I8, "i32": _lib.I32}
    assert _host_parts(ids[tin], ids[tout], M, N, K) == parts


def _choice(in_type, out_type, M, N, K, a_col=False, b_col=False, epilogue=_lib.EPILOGUE_RELU, epilogue_arg=0.0, batch=1, prologue_arg=0.0):
    """(variant, K slices) the library takes for dense, aligned operands (nothing is launched)."""
    ids = {"f16": _lib.F16, "bf16": _lib.BF16, "i8": _lib.I8, "f32": _lib.F32, "i32": _lib.I32, "i16": _lib.I16}
    L, h, v, ks, P = _lib.lib(), ctypes.c_int(-1), ctypes.c_int(), ctypes.c_int(), ctypes.c_void_p
    many = int(batch > 1)
    _lib.check(L.acc950_bind(ids[in_type], ids[out_type], batch, M, N, K, P(1 << 40), many * M * K, *((1, M) if a_col else (K, 1)), P(2 << 40), many * K * N, *((1, K) if b_col else (N, 1)),
                             P(3 << 40), many * M * N, N, 1, _lib.PROLOGUE_SET0, prologue_arg, epilogue, epilogue_arg, _lib.VARIANT_AUTO, 0, None, ctypes.byref(h)))
    try:
        _lib.check(L.acc950_bound_choice(h.value, ctypes.byref(v), ctypes.byref(ks)))
    finally:
        L.acc950_unbind(h.value)
    return v.value, ks.value


@pytest.mark.parametrize("in_type,out_type,batch,M,N,K,ops,short_k", [
    ("f16", "f16", 32, 2048, 2048, 128, "scale", True), ("f16", "f16", 1, 8192, 8192, 64, "relu", True), ("bf16", "f32", 1, 6352, 2952, 96, "relu", True), ("bf16", "bf16", 1, 51424, 4096, 128, "relu", True),
    ("f16", "f16", 1, 50176, 256, 128, "none", False), ("f16", "f16", 1, 69872, 256, 128, "none", True), ("f16", "f16", 1, 67168, 256, 64, "none", True),  # one column tile
    ("f16", "f16", 1, 36240, 384, 128, "relu", False), ("f16", "f16", 1, 36240, 384, 128, "scale", True), ("f16", "f16", 1, 46080, 384, 128, "relu", True),  # two, a little more than a round
    ("bf16", "f32", 1, 22592, 4864, 128, "relu", False), ("bf16", "f32", 1, 22592, 4864, 128, "scale", True), ("bf16", "f32", 1, 12288, 4864, 128, "relu", True),  # 440 and 239 MB of C
    ("bf16", "f32", 80, 992, 1024, 128, "none", True), ("i8", "i32", 1, 10624, 9728, 256, "relu", False), ("i8", "i16", 1, 10624, 9728, 256, "relu", True),
    ("i8", "i32", 1, 10624, 4864, 256, "relu/col", True), ("i8", "i32", 1, 9376, 9800, 256, "relu/col", True), ("i8", "i32", 1, 3792, 1352, 256, "none/col", True),  # not the four-wave kernel's
    ("bf16", "bf16", 1, 15072, 22256, 128, "none", True), ("bf16", "bf16", 1, 2656, 5144, 128, "none", True), ("f16", "f16", 1, 7264, 9592, 128, "relu", True),  # rows off 64-byte boundaries
    ("bf16", "bf16", 1, 5152, 1832, 96, "none", True), ("bf16", "bf16", 1, 3232, 1832, 96, "none", False), ("bf16", "bf16", 1, 560, 13512, 64, "none", True), ("i8", "i32", 1, 3232, 1832, 128, "none/col", True),  # ... two, one tile per CU
    ("f16", "f32", 1, 19904, 8240, 32, "none", False), ("f16", "f32", 1, 3904, 8240, 32, "none", True), ("f16", "f32", 160, 64, 1136, 96, "relu", True),  # on odd multiples of 64 bytes
    ("i8", "i32", 1, 10000, 9744, 128, "none", False), ("i8", "i32", 1, 5000, 9744, 128, "none", True), ("f16", "f16", 1, 20000, 8224, 64, "none", False), ("f16", "f16", 1, 20000, 8224, 128, "none", True),
])
def test_where_the_short_k_kernel_is_taken(in_type, out_type, batch, M, N, K, ops, short_k):
    """Both sides of the lines where another kernel is level or ahead (figures beside the rule)."""
    ops, _, b = ops.partition("/")
    epilogue, arg = {"none": (_lib.EPILOGUE_NONE, 0.0), "relu": (_lib.EPILOGUE_RELU, 0.0), "scale": (_lib.EPILOGUE_SCALE, 0.125)}[ops]
    assert (_choice(in_type, out_type, M, N, K, epilogue=epilogue, epilogue_arg=arg, batch=batch, b_col=b == "col")[0] == _lib.VARIANT_SHORT_K) == short_k


@pytest.mark.parametrize("in_type,M,N,K,tile,slices", [
    ("f16", 3296, 1088, 5026, "128x128", 1), ("f16", 3296, 1088, 5306, "256x256", 3),   # 234 tiles of 128 x 128: nearly a whole round
    ("f16", 1520, 1344, 3802, "256x256", 6),                                            # 132 of them
    ("bf16", 3713, 800, 4933, "256x256", 4), ("f16", 1046, 3061, 5162, "256x256", 4),   # rows of B off dwords; 60 large tiles
    ("i8", 447, 5145, 5765, "256x256", 6), ("i8", 447, 5145, 5764, "128x128", 1),       # rows of B off dwords, and on them
    ("i8", 5184, 736, 5790, "128x128", 1), ("i8", 5184, 736, 6002, "256x256", 4), ("i8", 644, 7700, 5155, "256x256", 2),
])
def test_large_tiles_in_slices_against_a_k_contiguous_b(in_type, M, N, K, tile, slices):
    """K has to be longer where the 128 x 128 tiles fill the chip in one round and rows of B are whole dwords apart."""
    v, ks = _choice(in_type, "i32" if in_type == "i8" else in_type, M, N, K, b_col=True)
    assert f"mfma {tile} " in _lib.variant_name(v) and "any-alignment" in _lib.variant_name(v) and ks == slices, (_lib.variant_name(v), ks)


def test_eager_call_passes_streams_and_falls_back_on_a_refusal_only(monkeypatch):
    """accera_amd.gemm_relu against a stand-in for the library: the raw stream as an int, a c_void_p or the current one; a recorded kernel that the library
    refuses makes way for its own choice, a launch that fails does not."""
    import struct
    import types

    import torch
    from accera_amd import gemm, tuned

    class Matrix:  # what the front end asks of a tensor
        shape, dtype, is_cuda, device = torch.Size((64, 64)), torch.float16, True, "cuda:0"
        def stride(self): return (64, 1)
        def dim(self): return 2
        def data_ptr(self): return 1 << 20
        def get_device(self): return 0

    calls, codes = [], []

    def packed(call):
        calls.append(struct.Struct("19qdqd3q").unpack(call)[-3:])   # variant, K slices, stream
        return codes.pop(0)

    monkeypatch.setattr(gemm._lib, "lib", lambda: types.SimpleNamespace(acc950_gemm_packed=packed, acc950_last_error=lambda: b"stand-in"))
    monkeypatch.setattr(tuned, "recorded", lambda *a: (7, 2))
    run = lambda **kw: gemm.gemm_relu(Matrix(), Matrix(), Matrix(), **kw)
    for stream, raw in ((5, 5), (ctypes.c_void_p(6), 6), (ctypes.c_void_p(None), 0), (0, 0)):
        codes[:] = [_lib.OK]
        run(stream=stream)
        assert calls.pop() == (7, 2, raw) and not calls
    for way in ((lambda device: 9), None):
        monkeypatch.setattr(gemm, "_raw_stream", way)
        monkeypatch.setattr(torch.cuda, "current_stream", lambda device: types.SimpleNamespace(cuda_stream=9))
        codes[:] = [_lib.OK]
        run()
        assert calls.pop() == (7, 2, 9)
    codes[:] = [_lib.UNSUPPORTED, _lib.OK]
    run(stream=5)
    assert calls == [(7, 2, 5), (_lib.VARIANT_AUTO, 0, 5)]
    calls.clear()
    codes[:] = [_lib.HIP_ERROR]
    with pytest.raises(_lib.Acc950Error):
        run(stream=5)
    assert calls == [(7, 2, 5)]
