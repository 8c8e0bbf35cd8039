"""CPU-side checks of the drop-in boundary: the shared library loads without a GPU, exports every
symbol the public header declares, and reports errors instead of computing without a device."""
import ctypes as C
import os
import subprocess
import sys
import sysconfig

import pytest

from warpdecode_amd import build, capi, synth


def test_exports_every_declared_symbol():
    lib = capi.load()
    declared = capi.declared_symbols()
    assert len(declared) >= 40
    missing = [s for s in declared if not hasattr(lib, s)]
    assert not missing, missing


@pytest.mark.parametrize("t", [synth.Q4_0, synth.Q8_0, synth.IQ4_NL, synth.IQ3_S, synth.IQ2_S])
def test_block_geometry(t):
    lib = capi.load()
    assert lib.wd_row_bytes(t, 2048) == synth.row_bytes(t, 2048)
    assert lib.wd_row_bytes(t, 2048 + 1) == 0
    assert lib.wd_tensor_bytes(t, 512, 2048) == 512 * synth.row_bytes(t, 2048)
    assert lib.wd_row_bytes(99, 2048) == 0


def test_argument_errors_are_reported():
    lib = capi.load()
    # geometry is validated before any device work, so these fail the same way with or without a GPU
    assert lib.wd_q8_k_quantize_f32(None, 100, None, None, None, None) == -1
    assert b"multiple of 256" in lib.wd_last_error()
    assert lib.wd_topk_softmax(None, 12, 2, 1.0, None, None, None) == -1
    assert b"multiple of 8" in lib.wd_last_error()
    assert lib.wd_gemv_q8_k_f32(synth.Q8_0, C.c_void_p(8), 4, 256, None, None, None, None, None) == -1
    with pytest.raises(capi.WdError):
        capi.call("wd_q8_0_quantize_f32", None, 33, None, None, None)


def test_profiler_switched_off_touches_nothing():
    """The site profiler's names follow the reference's numbering (src/qwen38_moe.cuh:296-352), and with the switch off
    its hooks are no-ops that need no device."""
    from warpdecode_amd import capi
    lib = capi.load()
    names = [lib.wd_profile_site_name(i).decode() for i in range(24)]
    assert names[0] == "moe.stage_total" and names[1] == "moe.routed_total" and names[2] == "moe.router_select"
    assert names[10] == "moe.acquire" and names[13] == "moe.batch.gate_up" and names[17] == "moe.batch.accum"
    assert names[20] == "moe.finish" and names[23] == "moe.mirror" and len(set(names)) == 24
    assert lib.wd_profile_site_name(24) == b"moe.fused.ab"
    assert lib.wd_profile_site_name(-1) == b"unknown" and lib.wd_profile_site_name(1000) == b"unknown"
    assert lib.wd_profile_enabled() == 0
    capi.call("wd_profile_begin", 0, None)
    capi.call("wd_profile_end", 0, None)
    capi.call("wd_profile_flush_token")
    st, tokens = capi.ProfileSiteStat(), C.c_ulonglong(7)
    capi.call("wd_profile_site", 0, C.byref(st), C.byref(tokens))
    assert (st.calls, st.recorded, st.dropped, st.host_ms, tokens.value) == (0, 0, 0, 0.0, 0)
    assert lib.wd_profile_begin(1000, None) != 0 and b"out of range" in lib.wd_last_error()
    need = lib.wd_profile_report(None, 0)
    buf = C.create_string_buffer(need + 1)
    assert lib.wd_profile_report(buf, need + 1) == need
    assert buf.value == b"[moe-profile] tokens=0 unit=ms_per_token\n"


SPAN = (C.c_uint8 * 4096)()
CALLS = [
    ("wd_q8_k_quantize_f32", None, 100, None, None, None, None), ("wd_q8_0_quantize_f32", C.c_void_p(8), 33, SPAN, 8, None),
    ("wd_topk_softmax", None, 12, 2, 1.0, None, None, None), ("wd_topk_softmax", None, 12, 2, 1, None, None, None),
    ("wd_topk_softmax", None, 12, 2, "1", None, None, None), ("wd_topk_softmax", None, 12.0, 2, 1.0, None, None, None),
    ("wd_topk_softmax", None, (1 << 32) + 12, -5, 1.0, None, None, None), ("wd_topk_softmax", True, 12, True, 1.0, None, -1, 1 << 70),
    ("wd_topk_softmax", C.byref(SPAN), C.c_int(12), 2, C.c_float(1), C.POINTER(C.c_uint8)(), None, None),
    ("wd_topk_softmax", b"x", 12, 2, 1.0, "x", None, None), ("wd_topk_softmax", None, 12, 2, 1.0, None, None),
    ("wd_topk_softmax", None, 12, 2, 1.0, None, None, None, None), ("wd_topk_softmax",), ("wd_no_such_thing", 1), (1, 2), (),
    ("wd_gemv_q8_k_f32", synth.Q8_0, C.c_void_p(8), 4, 256, None, None, None, None, None),
    ("wd_gemv_q8_0_f32", synth.Q8_0, SPAN, 0, 256, SPAN, None, 8, None, None), ("wd_gemv_q8_0_f32", synth.Q8_0, 1.5, 0, 256, SPAN, None, 8, None, None),
    ("wd_moe_scratch_create", C.byref(C.c_void_p()), 100, 512, 64, 8),
]


@pytest.mark.parametrize("args", CALLS, ids=lambda a: "-".join(str(x)[:8] for x in a[:1]) or "nothing")
def test_calls_without_ctypes_answer_as_with_it(args):
    """Every form of an argument is taken, or refused with the same words, on both ways to an entry point."""
    assert capi._fast is not None and capi.call is capi._fast.call, "the extension is not built"
    capi.load()

    def outcome(call):
        try:
            return call(*args)
        except Exception as e:   # noqa: BLE001 (whatever it is has to be alike)
            return type(e), str(e).replace("_call", "call")
    want = outcome(capi._call)
    assert want is not None and outcome(capi.call) == want


def test_arguments_arrive_as_with_ctypes():
    """What each form of an argument becomes: entry points that hand their own arguments back."""
    seen = []
    kind = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_int, C.c_float, C.c_void_p, C.c_void_p, C.c_void_p)
    stand_in = kind(lambda *a: seen.append(a) or 0)
    lib = capi.load()
    true_fn = lib.wd_topk_softmax
    rows = [(None, 8, 2, 1.5, SPAN, C.c_void_p(), C.c_void_p(77)), ((1 << 64) - 8, -3, (1 << 32) + 5, -0.0, True, -1, 1 << 63),
            (0, 2**31, -2**31, 1e300, None, (1 << 64) + 9, (C.c_void_p * 2)())]
    try:
        capi._fast.prepare(capi._call, capi.check, C.c_void_p, C.Array)
        capi._fast.bind("wd_topk_softmax", C.cast(stand_in, C.c_void_p).value)
        for r in rows:
            assert capi.call("wd_topk_softmax", *r) is None
            stand_in.argtypes = true_fn.argtypes
            stand_in(*r)
            assert repr(seen[-1]) == repr(seen[-2])
        with pytest.raises(ValueError):
            capi._fast.bind("wd_topk_softmax", 8)
    finally:
        capi._fast.prepare(capi._call, capi.check, C.c_void_p, C.Array)
        for name in capi._fast.names():
            capi._fast.bind(name, C.cast(getattr(lib, name), C.c_void_p).value)


FIRST_CALLS = """
import sys, threading, time
from warpdecode_amd import capi
real, gate, answers = capi.C.CDLL, threading.Barrier(8), []
def slow_load(path):    # every thread that gets this far is in the load together
    time.sleep(0.05)
    return real(path)
capi.C.CDLL = slow_load
def first():
    gate.wait()
    try:
        answers.append(capi.call("wd_topk_softmax", None, 12, 2, 1.0, None, None, None))
    except Exception as e:
        answers.append((type(e).__name__, str(e)))
threads = [threading.Thread(target=first) for _ in range(8)]
[t.start() for t in threads]
[t.join() for t in threads]
assert len(answers) == 8 and set(answers) == {answers[0]} and answers[0][0] == "WdError" and "multiple of 8" in answers[0][1], answers
"""
LOAD_AGAIN = """
from warpdecode_amd import capi
real = capi._fast
class FailsOnTheWay:
    bound = 0
    names, signature = staticmethod(real.names), staticmethod(real.signature)
    @classmethod
    def bind(cls, *a):
        if cls.bound == 3: raise MemoryError("on the way")
        cls.bound += 1
        real.bind(*a)
capi._fast = FailsOnTheWay
for _ in range(2):
    FailsOnTheWay.bound = 0
    try:
        capi.load()
        raise SystemExit("the load did not fail")
    except MemoryError:
        pass
capi._fast = real
assert capi.load() is capi.load()
"""


OTHER_PROTOTYPE = """
from warpdecode_amd import capi
real, bound = capi._fast, []
class OfOtherSources:
    names = staticmethod(real.names)
    signature = staticmethod(lambda name: "piizppp" if name == "wd_topk_softmax" else real.signature(name))
    bind = staticmethod(lambda *a: bound.append(a[0]) or real.bind(*a))
capi._fast = OfOtherSources
capi.load()
assert sorted(bound) == sorted(set(real.names()) - {"wd_topk_softmax"}), bound
try:
    capi.call("wd_topk_softmax", None, 12, 2, 1.0, None, None, None)
except capi.WdError as e:
    assert "multiple of 8" in str(e)
"""


@pytest.mark.parametrize("program", [FIRST_CALLS, LOAD_AGAIN, OTHER_PROTOTYPE], ids=["several_threads", "after_a_failure", "another_prototype"])
def test_first_load(program):
    """In a process of its own: the first calls of several threads all get the library's answer, a load that failed can be tried again, and
    an entry point that the extension knows with other arguments is called through ctypes."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = subprocess.run([sys.executable, "-c", program], cwd=root, capture_output=True, text=True, timeout=120)
    assert got.returncode == 0, got.stderr


def test_extension_belongs_to_this_interpreter_and_these_prototypes():
    assert capi._fast.__file__ == build.FAST and build.FAST.endswith(sysconfig.get_config_var("EXT_SUFFIX"))
    assert len(capi._fast.names()) == 17
    for name in capi._fast.names():
        res, args = capi._SIGS[name]
        assert res is capi.i32 and [capi._CODES[a] for a in args] == list(capi._fast.signature(name)), name


@pytest.mark.parametrize("missing", ["header", "compiler"])
def test_a_machine_that_cannot_build_the_extension(monkeypatch, tmp_path, capfd, missing):
    """It is left out, with a word on stderr and without an older one staying behind."""
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "FAST", str(tmp_path / "_fast.old"))
    for name in ("_fast.old", "_fast.so"):
        (tmp_path / name).write_bytes(b"of older sources")
    if missing == "header":
        monkeypatch.setattr(build.sysconfig, "get_paths", lambda: {"include": str(tmp_path)})
    else:
        monkeypatch.setenv("PATH", str(tmp_path))
    assert build.build_fast() is None
    assert not os.listdir(tmp_path) and "not built" in capfd.readouterr().err
