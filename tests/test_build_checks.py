"""The build's reader of the compiler's resource remarks (accera_amd/csrc/check_resources.py): what it has to notice, in
the two forms in which compilers write the remarks, and that a file it does not understand is not taken for a clean one."""
import importlib.util
import os

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "accera_amd", "csrc")
W4 = "_ZN6acc95020gemm_mfma16w4_kernelINS_14Mfma16W4ConfigILi0ELb1EEEEEvPKv"


def _check():
    spec = importlib.util.spec_from_file_location("check_resources", os.path.join(CSRC, "check_resources.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def _remarks(form, kernels):
    lines = []
    for name, scratch in kernels:
        for body in (f"Function Name: {name}", "    VGPRs: 256", f"    ScratchSize [bytes/lane]: {scratch}", "    VGPRs Spill: 3"):
            lines.append(form.format(body) + " [-Rpass-analysis=kernel-resource-usage]")
    return "\n".join(lines) + "\n"


@pytest.mark.parametrize("form", ["remark: ./gemm_mfma.h:512:0: {}", "./gemm_mfma.h:512:0: remark: {}"])
def test_scratch_of_a_four_wave_kernel_fails_the_build(form, tmp_path, capsys):
    check, path = _check(), tmp_path / "unit.resources.txt"
    path.write_text(_remarks(form, [("_ZN6acc9505otherEv", 88), (W4, 0)]))
    assert check.main([str(path)]) == 0
    path.write_text(_remarks(form, [(W4, 16)]))
    assert check.main([str(path)]) == 1
    assert "16 bytes of scratch" in capsys.readouterr().err


def test_a_file_without_a_known_kernel_fails_the_build(tmp_path, capsys):
    check, path, listing = _check(), tmp_path / "unit.resources.txt", tmp_path / "unit.s"
    listing.write_text(f"{W4}:\n\ts_endpgm\n.Lfunc_end0:\n")
    path.write_text("remark made of something else\n")
    assert check.main([str(listing)]) == 0
    assert check.main([str(path), str(listing)]) == 1
    assert "unit.resources.txt" in capsys.readouterr().err


def _staged(edge, any_alignment=True):
    return (f"_ZN6acc95016gemm_mfma_kernelINS_10MfmaConfigILi2ELi{edge}ELi{edge}ELi2ELi2ELb1ELb0ELb0ELb1ELi128ELi2ELb0ELb0ELb{int(any_alignment)}ELb0EEEEEvPKv")


@pytest.mark.parametrize("edge,vgprs,scratch,fails", [(64, 128, 0, False), (64, 132, 0, True), (64, 128, 8, True), (128, 222, 0, False), (128, 222, 16, True),
                                                      (256, 256, 20, False), (256, 254, 68, True)])
def test_registers_and_scratch_of_the_register_staged_kernels(edge, vgprs, scratch, fails, tmp_path, capsys):
    """A CU holds four workgroups of the 64 x 64 tiles (the kernel choice counts on it), and none of these kernels may spill
    more than they do."""
    check, path = _check(), tmp_path / "unit.resources.txt"
    form = "remark: ./gemm_mfma.h:512:0: {}"
    own = _remarks(form, [(_staged(edge), scratch)]).replace("VGPRs: 256", f"VGPRs: {vgprs}")
    path.write_text(_remarks(form, [(W4, 0)]) + own)
    assert check.main([str(path)]) == int(fails)
    assert not fails or f"{vgprs} vector registers" in capsys.readouterr().err


SHORT_K = "_ZN6acc95019gemm_short_k_kernelINS_12ShortKConfigILi0ELb1ELb1ELi4ELi4EEEEEvPKv"


@pytest.mark.parametrize("name,scratch,fails", [
    (SHORT_K, 0, False), (SHORT_K, 4, True),
    # 32x32-shape kernels with direct fills: fp16, int8
    (_staged(256).replace("ELb0ELb1ELi128ELi2E", "ELb1ELb0ELi64ELi4E").replace("ConfigILi2E", "ConfigILi0E"), 0, False),
    (_staged(256).replace("ELb0ELb1ELi128ELi2E", "ELb1ELb0ELi64ELi4E").replace("ConfigILi2E", "ConfigILi0E"), 68, True),
    (_staged(256).replace("ELb0ELb1ELi128ELi2E", "ELb1ELb0ELi64ELi4E"), 76, False),
    (_staged(256).replace("ELb0ELb1ELi128ELi2E", "ELb1ELb0ELi64ELi4E"), 276, True),
    (_staged(256).replace("ConfigILi2E", "ConfigILi1E"), 20, True),
])
def test_scratch_of_the_other_kernels(name, scratch, fails, tmp_path, capsys):
    check, path = _check(), tmp_path / "unit.resources.txt"
    form = "remark: ./gemm_mfma.h:512:0: {}"
    path.write_text(_remarks(form, [(W4, 0), (name, scratch)]))
    assert check.main([str(path)]) == int(fails)
    assert not fails or f"{scratch} bytes of scratch" in capsys.readouterr().err
    path.write_text(_remarks(form, [(SHORT_K, 0)]))
    assert check.main([str(path)]) == 0    # (a unit of short-K kernels is understood)
