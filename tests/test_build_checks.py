"""Device-code checks that run at build time (no GPU needed: hipcc cross-compiles).

The GEMMs and the wide attention stage operands with buffer loads that write LDS directly;
the counted wait before the MFMAs that read them is correct only while the compiler keeps
the issue order the source pins. build_lib.check_kblock_waits (the skinny GEMM),
check_chunk_waits (kernels whose waves keep their copies to themselves) and check_step_waits
(kernels that share them behind a barrier) re-derive that from the generated assembly; these
tests show that they pass on the real kernels and reject a wait that would let the MFMAs read
LDS too early.
"""
import re
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "flash-vla_amd"))
import build_lib  # noqa: E402

pytestmark = pytest.mark.skipif(not os.path.exists(build_lib.HIPCC) and not shutil.which("hipcc"),
                                reason="needs hipcc")


def _asm(name):
    src = os.path.join(build_lib.CSRC, name)
    res = subprocess.run([build_lib.HIPCC, *build_lib.FLAGS, "--cuda-device-only", "-S", src,
                          "-o", "-"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    return res.stdout


@pytest.fixture(scope="module")
def gemm_asm():
    return _asm("pi0_gemm.hip")


@pytest.fixture(scope="module")
def encoder_asm():
    return _asm("pi0_encoder.hip")


def test_kblock_waits_hold(gemm_asm):
    assert "skinny_gemm_kernel" in gemm_asm
    assert build_lib.check_kblock_waits(gemm_asm) == []


# the gate kernel (x rows then weights per k-block), the QKV kernel (all weights first),
# each also with 56 of the 64 rows staged
@pytest.mark.parametrize("name", [
    "_ZN3pi018skinny_gemm_kernelILi4ELb1ELi8ELi4ELin1ELi64EEEvNS_8GemmArgsE",
    "_ZN3pi018skinny_gemm_kernelILi4ELb1ELi8ELi4ELin1ELi56EEEvNS_8GemmArgsE",
    "_ZN3pi018skinny_gemm_kernelILi3ELb0ELi8ELi4ELi4ELi64EEEvNS_8GemmArgsE",
    "_ZN3pi018skinny_gemm_kernelILi3ELb0ELi8ELi4ELi4ELi56EEEvNS_8GemmArgsE"])
def test_kblock_waits_reject_a_loose_wait(gemm_asm, name):
    start = gemm_asm.index(name + ":")
    body = gemm_asm[start:gemm_asm.index("s_endpgm", start)]
    first = body.index("s_waitcnt vmcnt(", body.index(" lds\n"))   # first k-block wait
    loose = body[:first] + "s_waitcnt vmcnt(60)" + body[body.index(")", first) + 1:]
    assert build_lib.check_kblock_waits(gemm_asm.replace(body, loose)) == [name]


def _with_wait(asm, name, nth, n):
    """`asm` with the nth vmcnt wait of kernel `name` behind its first LDS copy made vmcnt(n)."""
    start = asm.index(name + ":")
    end = asm.index("s_endpgm", start)
    first = asm.index(" lds\n", start)
    w = list(re.finditer(r"vmcnt\(\d+\)", asm[first:end]))[nth]
    return asm[:first + w.start()] + f"vmcnt({n})" + asm[first + w.end():]


def test_chunk_waits_hold(gemm_asm, encoder_asm):
    """The gate kernel is known to wait for all four chunks before each row block's first: the
    compiler adds that wait where it cannot tell the slot refilled last from the one read next."""
    loose, full = build_lib.check_chunk_waits(encoder_asm)
    assert loose == [] and full == []
    loose, full = build_lib.check_chunk_waits(gemm_asm)
    assert loose == [] and all("gate_stream_kernel" in k for k in full)


@pytest.mark.parametrize("name,nth", [
    ("_ZN3pi017rows32_res_kernelILi16EEEvNS_8TileArgsEii", 1),
    ("_ZN3pi017rows32_res_kernelILi32EEEvNS_8TileArgsEii", 0),
    ("_ZN3pi017rows32_res_kernelILi32EEEvNS_8TileArgsEii", 5),
    ("_ZN3pi017qkv_rows32_kernelILi5EEEvNS_8GemmArgsE", 2),
    ("_ZN3pi018gate_stream_kernelILi2EEEvNS_8GemmArgsE", None),
    ("_ZN3pi018gate_stream_kernelILi4EEEvNS_8GemmArgsE", None)])
def test_chunk_waits_reject_a_changed_wait(gemm_asm, encoder_asm, name, nth):
    asm = gemm_asm if name + ":" in gemm_asm else encoder_asm
    if nth is None:              # every chunk is waited for twice there: loosen all waits
        start = asm.index(name + ":")
        end = asm.index("s_endpgm", start)
        asm = asm[:start] + re.sub(r"vmcnt\(\d+\)", "vmcnt(60)", asm[start:end]) + asm[end:]
        assert build_lib.check_chunk_waits(asm)[0] == [name]
        return
    assert build_lib.check_chunk_waits(_with_wait(asm, name, nth, 60))[0] == [name]
    assert name in build_lib.check_chunk_waits(_with_wait(asm, name, 0, 0))[1]


def test_step_waits_hold(encoder_asm):
    for kernel in build_lib._SHARED_STEPS:
        assert any(True for _ in build_lib._kernels(encoder_asm, kernel)), kernel
    assert build_lib.check_step_waits(encoder_asm) == []


@pytest.mark.parametrize("name,nth", [
    ("_ZN3pi016tile_gemm_kernelILi192ELi32ELi4ELi5ELb0ELi1ELi0EEEvNS_8TileArgsE", 0),
    ("_ZN3pi017block_gemm_kernelILi4ELi2ELi2ELi4ELi3ELb1EEEvNS_8TileArgsE", 0),
    ("_ZN3pi017block_gemm_kernelILi4ELi2ELi2ELi4ELi3ELb1EEEvNS_8TileArgsE", 3),
    ("_ZN3pi017block_gemm_kernelILi4ELi2ELi3ELi4ELi3ELb1EEEvNS_8TileArgsE", 2),
    ("_ZN3pi020enc_attn_wide_kernelENS_11EncAttnArgsE", 0),
    ("_ZN3pi020enc_attn_wide_kernelENS_11EncAttnArgsE", 1)])
def test_step_waits_reject_a_changed_wait(encoder_asm, name, nth):
    assert build_lib.check_step_waits(_with_wait(encoder_asm, name, nth, 60)) == [name]
    start = encoder_asm.index(name + ":")        # the wait for the reads of the slot filled next
    if "tile_gemm" not in name:
        body = encoder_asm[start:]
        assert build_lib.check_step_waits(
            encoder_asm[:start] + re.sub(r"(vmcnt\(\d+\)) lgkmcnt\(0\)", r"\1", body, count=1)) == [name]


def test_activation_copies_stay_inside_the_range_check(gemm_asm, encoder_asm):
    """Rows past M and the columns past a padded K's end are zeros because the copy's whole
    offset is the lane's (see build_lib.unchecked_copies)."""
    assert "block_gemm_kernel" in encoder_asm and "rows32_res_kernel" in encoder_asm
    assert build_lib.unchecked_copies(encoder_asm) == []
    assert build_lib.unchecked_copies(gemm_asm) == []
    fake = "_ZN3pi07k_looseEv:\n\tbuffer_load_dwordx4 v1, s[0:3], s9 offen lds\n\ts_endpgm\n"
    assert build_lib.unchecked_copies(fake) == ["_ZN3pi07k_looseEv"]
    assert build_lib.unchecked_copies(fake.replace("s9", "0")) == []


def test_no_packed_fp32(gemm_asm):
    assert not build_lib._PACKED_FP32.search(gemm_asm)


def test_no_kernel_uses_scratch():
    """Every kernel runs without a scratch segment: a runtime-indexed kernel argument
    (copied to the stack) or a register spill shows up here before it shows up as a
    slowdown on the GPU."""
    src = os.path.join(build_lib.CSRC, "pi0_attention.hip")
    res = subprocess.run([build_lib.HIPCC, *build_lib.FLAGS, "--cuda-device-only", "-S", src,
                          "-o", "-"], capture_output=True, text=True)
    assert res.returncode == 0, res.stderr
    assert "attn_kernel" in res.stdout
    assert build_lib.scratch_kernels(res.stdout) == []
    fake = ("\t.amdhsa_kernel k_spills\n\t\t.amdhsa_private_segment_fixed_size 192\n"
            "\t.end_amdhsa_kernel\n\t.amdhsa_kernel k_clean\n"
            "\t\t.amdhsa_private_segment_fixed_size 0\n\t.end_amdhsa_kernel\n")
    assert build_lib.scratch_kernels(fake) == ["k_spills"]
