"""What the compiler gave the kernels that several workgroups of a compute unit depend on: vector registers, scratch and spills, from
the metadata of the library that was built here.  (A compute unit has four SIMDs of 512 registers per lane: six waves on each need at most 80.)"""
import os
import re
import subprocess

import pytest

from warpdecode_amd import build

BIN = "/opt/rocm/llvm/bin/"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """name -> (vector registers, bytes of scratch per lane, spilled vector registers)"""
    if not os.path.exists(BIN + "clang-offload-bundler"):
        pytest.skip("no LLVM tools")
    if not os.path.exists(build.LIB):
        build.build()
    d = tmp_path_factory.mktemp("co")
    fat, co = str(d / "fatbin"), str(d / "co")
    subprocess.check_call([BIN + "llvm-objcopy", "--dump-section", ".hip_fatbin=" + fat, build.LIB, os.devnull])
    subprocess.check_call([BIN + "clang-offload-bundler", "--type=o", "--unbundle", "--input=" + fat, "--output=" + co,
                           "--targets=hipv4-amdgcn-amd-amdhsa--gfx950"])
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
