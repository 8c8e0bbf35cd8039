"""The kernels of the library that was built here, as they came out of the compiler.  Vector registers, scratch and spills where several workgroups are meant to
share a compute unit (it has four SIMDs of 512 registers per lane: six waves on each need at most 80); and the statements in assembly whose wait
states the compiler does not know."""
import os
import re
import subprocess

import pytest

from warpdecode_amd import build

BIN = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def code_object(tmp_path_factory):
    if not os.path.exists(BIN + "clang-offload-bundler"):
        pytest.skip("no LLVM tools")
    if not os.path.exists(build.LIB):
        build.build()
    d = tmp_path_factory.mktemp("co")
    fat, co = str(d / "fatbin"), str(d / "co")
    subprocess.check_call([BIN + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, build.LIB, os.devnull])
    subprocess.check_call([BIN + "clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + co,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
    return co


@pytest.fixture(scope="module")
def kernels(code_object):
    """name -> (vector registers, bytes of scratch per lane, spilled vector registers)"""
    co = code_object
    notes = subprocess.run([BIN + "llvm-readelf", "--notes", co], check=True, capture_output=True, text=True).stdout
    field = lambda text, name: int(re.search(r"\.%s:\s+(\d+)" % name, text).group(1))
    out = {}
    for text in notes.split("  - .agpr_count")[1:]:
        name = re.search(r"\.name:\s+(\S+)", text).group(1)
        out[name] = (field(text, "vgpr_count"), field(text, "private_segment_fixed_size"), field(text, "vgpr_spill_count"))
    assert len(out) > 100
    return out


def _kernel(kernels, name, *args):
    """The instantiation of wd::`name` with these template arguments (the others as they come)."""
    mangled = "_ZN2wd%d%sI%s" % (len(name), name, "".join("Lb%dE" % a if isinstance(a, bool) else "Li%dE" % a for a in args))
    found = [v for n, v in kernels.items() if n.startswith(mangled)]
    assert len(found) == 1, (mangled, len(found))
    return found[0]


@pytest.mark.parametrize("args", [(0, 4, False, False, False, False), (1, 4, False, False, False, False),
                                  (0, 3, False, False, False, True, False), (1, 3, False, False, False, True, False)])
def test_two_workgroups_of_down_projections_fit_a_compute_unit(kernels, args):
    vgprs, scratch, spills = _kernel(kernels, "k_layer_c8", *args)
    assert vgprs <= 80 and scratch == 0 and spills == 0, (vgprs, scratch, spills)


@pytest.mark.parametrize("kind", [0, 1])
def test_two_workgroups_of_sixteen_waves_fit_a_compute_unit(kernels, kind):
    vgprs, scratch, spills = _kernel(kernels, "k_layer_c8", kind, 3, False, False, False, False, False)
    assert vgprs <= 64 and scratch == 0 and spills == 0, (vgprs, scratch, spills)


def test_spills_of_the_token_batch_at_ten_super_blocks(kernels):
    """Three workgroups per compute unit, bought with a few spills: not with more than when the figures beside the kernel were taken."""
    vgprs, scratch, spills = _kernel(kernels, "k_tokens_ab", 22, 4, 10)
    assert vgprs <= 80 and scratch <= 24 and spills <= 5, (vgprs, scratch, spills)


def test_scalar_operands_of_the_look_ups_come_from_their_own_statement(code_object):
    """A vector instruction that reads a scalar register needs two wait states behind a vector instruction that writes it.  The compiler keeps them
    for its own instructions, not for those of a statement in assembly: the byte and half-word selects of the IQ look-ups
    find their constant written by a scalar instruction right ahead of the two that use it, whatever the compiler puts in front."""
    dis = subprocess.Popen([BIN + "llvm-objdump", "-d", "--no-show-raw-insn", code_object], stdout=subprocess.PIPE, text=True)
    selects, before = 0, ["", ""]
    for line in dis.stdout:
        text = line.split("//")[0].strip()
        if text.startswith(("v_and_b32_sdwa", "v_lshlrev_b32_sdwa")):
            scalar = re.search(r", (s\d+), ", text)
            if scalar:
                selects += 1
                wrote = re.compile(r"(s_movk_i32|s_mov_b32) %s, " % scalar.group(1))
                assert any(wrote.match(b) for b in before), (before, text)
        before = [before[1], text]
    assert dis.wait() == 0 and selects > 1000
