"""The build's scratch guard: hipcc's kernel-resource remarks are parsed per
kernel, and the decode kernels' name patterns select what must not use
scratch memory (CPU)."""

from __future__ import annotations

import re

import pytest

from breeze_amd import build as B

_TAG = " [-Rpass-analysis=kernel-resource-usage]"


def _remarks(name: str, vgpr: int, scratch: int) -> str:
    lines = [
        f"Function Name: {name}",
        "    TotalSGPRs: 64",
        f"    VGPRs: {vgpr}",
        "    AGPRs: 0",
        f"    ScratchSize [bytes/lane]: {scratch}",
        "    Occupancy [waves/SIMD]: 4",
    ]
    return "".join(f"csrc/x.hip:12:1: remark: {l}{_TAG}\n" for l in lines)


def test_parse_remarks():
    text = (
        "csrc/x.hip:3:5: warning: something unrelated\n"
        + _remarks("_ZN2bz9gemv_mfmaILi0ELi4ELi1ELi4ELb0EEEvNS_10GemvParamsE", 73, 32)
        + _remarks("_ZN2bz15head_f32_kernelILi1ELi8EEEvPKfS2_iiPfi", 40, 0)
    )
    got = B.kernel_resources(text)
    assert got == [
        ("_ZN2bz9gemv_mfmaILi0ELi4ELi1ELi4ELb0EEEvNS_10GemvParamsE", 73, 32),
        ("_ZN2bz15head_f32_kernelILi1ELi8EEEvPKfS2_iiPfi", 40, 0),
    ]


def _checked(name: str) -> bool:
    return any(re.search(t, name) for t in B.NO_SCRATCH)


# one instance of every covered kernel, as compiled
COVERED = (
    "_ZN2bz12gemv_persistILi0ELi1ELi1ELi16ELb0EEEvPKtPKhPKvS2_iiiiiiNS_10GemvParamsE",
    "_ZN2bz9gemv_mfmaILi0ELi1ELi1ELi16ELb0EEEvPKtPKhPKvS2_iiiiiiNS_10GemvParamsE",
    "_ZN2bz10gemv_i8mmaILi0ELi1ELi1ELi2ELb0EEEvPKtPKhPKvS2_iiiiiiNS_10GemvParamsEi",
    "_ZN2bz9gemv_tileILi0ELi1ELi1ELi2EEEvPKtPKhPKviiiiiiiiNS_10TileParamsE",
    "_ZN2bz11gemv_streamILi4ELi1ELi10EEEvPKhPKtS4_iiiiiiiNS_12StreamParamsE",
    "_ZN2bz9gemv_wideILi4ELi1ELi2ELi0EEEvPKhPKtS4_iiiiiiiiNS_12StreamParamsE",
    "_ZN2bz10gemv_panelILi4ELi1ELi1ELi10EEEvPKhPKtiiiiiiiiNS_11PanelParamsE",
    "_ZN2bz9gemv_rowsILi1ELi1ELi2ELb0EEEvPKtPKhS2_iiiiiiNS_10GemvParamsE",
    "_ZN2bz9gemv_slabILi10EEEvPKhPKtiiiiiiNS_12StreamParamsE",
    "_ZN2bz10gemm_tiledILi4ELi2ELi1EEEvNS_10GemmParamsE",
    "_ZN2bz15head_f32_kernelILi1ELi1ELi0ELb0EEEvPKfliS2_liPKlliPflNS_8HeadNormE",
    "_ZN2bz12_GLOBAL__N_117sample_cfg_kernelENS0_12SampleParamsE",
    "_ZN2bz18step_tables_kernelIfEEviiPKlS2_fPT_S2_PKvifS4_S4_",
    "_ZN2bz21qkv_rope_cache_kernelEPKtliiiS1_S1_fPKvS3_blPKlPfPvS7_ibPl",
    "_ZN2bz9attn_bf16ILi1ELi16ELb0ELi8EEEvPKvS2_S2_PKlPvS5_ijNS_10AttnParamsE",
)


def test_patterns_cover_the_decode_kernels():
    for name in COVERED:
        assert _checked(name), name
    # fp32 caches and D = 512 are allowed scratch
    for name in (
        "_ZN2bz11attn_kernelILi4ELi16ELb1ELb0EEEvPKvS2_S2_PKlPvS5_iiNS_10AttnParamsE",
        "_ZN2bz11attn_kernelILi8ELi4ELb0ELb1EEEvPKvS2_S2_PKlPvS5_iiNS_10AttnParamsE",
    ):
        assert not _checked(name), name


def test_scratch_and_patterns_without_a_kernel_fail_the_build():
    kernels = [(name, 64, 0) for name in COVERED]
    B.check_scratch(kernels)
    for i, name in enumerate(COVERED):
        with pytest.raises(RuntimeError, match="no compiled kernel"):
            B.check_scratch(kernels[:i] + kernels[i + 1:])
        with pytest.raises(RuntimeError, match="scratch"):
            B.check_scratch(kernels[:i] + [(name, 64, 16)] + kernels[i + 1:])
