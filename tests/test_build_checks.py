"""CPU checks of the build's assembly checks: the 4x4x4 MFMA chains of
qmv_b4.hip are inline assembly, so mlxcel_amd.build.check_b4_mfma_chains
guards their register ties and wait states.  A well-formed chain passes and
each planted mistake is caught; the built library's own assembly (when
present) passes.  And the build itself: nothing unchecked is put in place, and
a machine without torch or g++ still gets a checked library."""
import os
import subprocess
import sys

import pytest

from mlxcel_amd import build as B

GOOD = """\
kernel:
\tv_perm_b32 v45, s0, v3, v45
\t;;#ASMSTART
\ts_nop 1
\tv_mfma_f32_4x4x4_16b_bf16 v[2:5], v[30:31], v[12:13], 0
\t;;#ASMEND
\tv_fma_f32 v7, v29, v26, 0
\ts_nop 1
\tv_mfma_f32_4x4x4_16b_bf16 v[2:5], v[14:15], v[32:33], v[2:5]
\ts_nop 0
\ts_nop 7
\ts_nop 7
\tv_fmac_f32_e32 v7, v28, v3
\ts_endpgm
"""


def test_good_chain_passes():
    assert B.check_b4_mfma_chains(GOOD) == 2


@pytest.mark.parametrize("old,new,msg", [
    ("v[2:5], v[30:31], v[12:13], 0", "v[2:5], v[4:5], v[12:13], 0", "overlaps"),
    ("v[32:33], v[2:5]", "v[32:33], v[6:9]", "neither 0 nor|wait states"),
    ("\ts_nop 1\n\tv_mfma_f32_4x4x4_16b_bf16 v[2:5], v[14:15]", "\tv_mfma_f32_4x4x4_16b_bf16 v[2:5], v[14:15]",
     "not s_nop"),
    ("\ts_nop 7\n\ts_nop 7\n", "\ts_nop 7\n", "wait states"),
    ("\ts_nop 7\n\ts_nop 7\n\tv_fmac", "\ts_cbranch_scc1 .LBB0_2\n\ts_nop 7\n\ts_nop 7\n\tv_fmac", "wait states"),
])
def test_planted_mistakes_are_caught(old, new, msg):
    bad = GOOD.replace(old, new, 1)
    assert bad != GOOD
    with pytest.raises(RuntimeError, match=msg):
        B.check_b4_mfma_chains(bad)


def test_no_mfma_is_an_error():
    with pytest.raises(RuntimeError, match="no 4x4x4 MFMA"):
        B.check_b4_mfma_chains("kernel:\n\ts_endpgm\n")


@pytest.mark.skipif(not os.path.exists(B.B4_ASM), reason="library not built here (no qmv_b4 assembly)")
def test_built_assembly_passes():
    assert B.check_b4_mfma_chains(open(B.B4_ASM).read()) > 0


@pytest.fixture
def stub_build(monkeypatch, tmp_path):
    """build() with its compilers replaced by ones that only create their output."""
    for name, file in (("LIB", "lib.so"), ("NATIVE", "native.so"), ("BENCH_LIB", "bench.so"), ("BUILD", "_build")):
        monkeypatch.setattr(B, name, str(tmp_path / file))

    def run(cmd, **kw):
        out = cmd[cmd.index("-o") + 1]
        open(out, "w").write(os.path.basename(cmd[0]))
        return subprocess.CompletedProcess(cmd, 0, "", "")

    monkeypatch.setattr(B.subprocess, "run", run)
    monkeypatch.setattr(B, "_verify_group_ring_waits", lambda: None)
    monkeypatch.setattr(B, "_verify_b4_mfma_chains", lambda: None)
    monkeypatch.setattr(B.shutil, "which", lambda name: name)
    return monkeypatch


def test_a_failed_check_leaves_no_library(stub_build):
    def bad():
        raise RuntimeError("planted")

    stub_build.setattr(B, "_verify_b4_mfma_chains", bad)
    with pytest.raises(RuntimeError, match="planted"):
        B.build(verbose=False)
    assert not os.path.exists(B.LIB) and not os.path.exists(B.NATIVE)


@pytest.mark.parametrize("missing", ["torch", "g++", "headers"])
def test_the_library_is_built_without_the_native_module(stub_build, missing):
    if missing == "torch":
        stub_build.setitem(sys.modules, "torch", None)  # import torch raises ImportError
    else:
        run = B.subprocess.run

        def no_gxx(cmd, **kw):
            if cmd[0] != "g++":
                return run(cmd, **kw)
            if missing == "g++":
                raise FileNotFoundError("g++")
            return subprocess.CompletedProcess(cmd, 1, "", "no such header")

        stub_build.setattr(B.subprocess, "run", no_gxx)
    open(B.NATIVE, "w").write("stale")
    with pytest.warns(UserWarning, match="ctypes"):
        B.build(verbose=False)
    assert os.path.exists(B.LIB) and os.path.exists(B.BENCH_LIB) and not os.path.exists(B.NATIVE)


def test_everything_present_builds_everything(stub_build):
    B.build(verbose=False)
    assert os.path.exists(B.LIB) and os.path.exists(B.BENCH_LIB) and os.path.exists(B.NATIVE)
