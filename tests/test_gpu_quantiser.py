"""The short form of the activations' Q8_0 quantiser (dispatch C) against the general one, bit for bit: every quotient of its range, and blocks at
the edges of that range, with ties, zeros, infinities and NaN."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "device", "libtest_quantiser.so")


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.init()
    return gpu_util


@pytest.fixture(scope="module")
def lib():
    if not os.path.exists(LIB):
        from warpdecode_amd import build
        build.build_device_test()
    return C.CDLL(LIB)


@pytest.fixture(scope="module")
def quant_range(lib):
    lo, span = C.c_uint32(), C.c_uint32()
    lib.test_range(C.byref(lo), C.byref(span))
    return lo.value, span.value


def test_every_quotient_of_the_range(g, lib, quant_range):
    """127 / a and a / 127 for every a from 2^-100 to 2^100, both included: 1,677,721,601 floats."""
    lo, span = quant_range
    bits = lambda v: int(np.float32(v).view(np.uint32))
    assert lo == bits(2.0 ** -100) and lo + span == bits(2.0 ** 100) and span + 1 == 1677721601
    wrong = g.empty(4, np.int32)
    assert lib.test_quotients(C.c_uint32(lo), C.c_uint32(span + 1), g.ptr(wrong)) == 0
    g.sync()
    w = g.host(wrong, np.uint32)
    assert w[0] == 0 and w[1] == 0, [hex(v) for v in w]


def _steps(rng):
    """(name, 512 values, whether the step has to take the general form; None: either)."""
    base = rng.normal(0, 1, 512).astype(np.float32)
    yield "ordinary", base, False
    for e in (-99, -60, -1, 0, 30, 99):
        yield "scaled", np.ldexp(base / np.abs(base).max(), e).astype(np.float32).repeat(1), None
    low, high = np.float32(2.0 ** -100), np.float32(2.0 ** 100)
    up, down = np.float32(np.inf), np.float32(0)
    for name, top, general in (("low", low, False), ("above low", np.nextafter(low, up), False), ("below low", np.nextafter(low, down), True),
                               ("high", high, False), ("below high", np.nextafter(high, down), False), ("above high", np.nextafter(high, up), True)):
        for sign in (1, -1):
            v = (rng.uniform(-1, 1, 512).astype(np.float32) * top * np.float32(0.999)).astype(np.float32)
            v[5::32] = top * np.float32(sign)                      # every block's largest
            yield name, v, general
            w = base.copy()
            w[64:96] = v[64:96]                                    # one such block among ordinary ones
            yield name + ", one block", w, general
    # quants at and around ties, and at +-127: a block whose largest is 127 / 2^j has the inverse scale 2^j
    for j in (0, 3, -5):
        for off in (0.0, 2.0 ** -17, -2.0 ** -17):
            v = np.ldexp(rng.integers(-126, 126, 512).astype(np.float32) + np.float32(0.5 + off), -j).astype(np.float32)
            v[::32] = np.ldexp(np.float32(127), -j) * rng.choice([-1, 1], 16).astype(np.float32)
            yield "ties", v, False
    for value in (0.0, -0.0, 2.0 ** -149, 2.0 ** -126, 3e38, np.inf, -np.inf, np.nan):
        for where in (slice(100, 101), slice(96, 128), slice(0, 512)):
            v = base.copy()
            v[where] = np.float32(value)
            small = abs(value) < 1e-30
            yield "value %r" % value, v, True if not small else where.stop - where.start >= 32
    payload = np.array([0x7fc00000, 0xffc00000, 0x7f800001, 0xff800001, 0x7fffffff, 0xffffffff], np.uint32).view(np.float32)
    for nan in payload:
        v = base.copy()
        v.view(np.uint32)[300] = np.asarray(nan).view(np.uint32)
        yield "nan", v, True


def test_steps_of_both_forms(g, lib):
    rng = np.random.default_rng(20261205)
    steps = list(_steps(rng))
    for i in range(2000):   # ordinary blocks of magnitudes of their own
        v = (rng.normal(0, 1, (16, 32)) * 2.0 ** rng.uniform(-95, 95, (16, 1))).astype(np.float32).reshape(-1)
        steps.append(("random", v, False))
    x, n = np.concatenate([v for _, v, _ in steps]), len(steps)
    dx, general = g.dev(x), g.empty(n, np.int32)
    qs, qg = g.empty(512 * n, np.int8), g.empty(512 * n, np.int8)
    d, dg = g.empty(16 * n, np.uint16), g.empty(16 * n, np.uint16)
    assert lib.test_steps(g.ptr(dx), n, g.ptr(qs), g.ptr(d), g.ptr(qg), g.ptr(dg), g.ptr(general)) == 0
    g.sync()
    qs, qg, d, dg = g.host(qs).reshape(n, 512), g.host(qg).reshape(n, 512), g.host(d, np.uint16).reshape(n, 16), g.host(dg, np.uint16).reshape(n, 16)
    general = g.host(general)
    for i, (name, v, expect) in enumerate(steps):
        assert np.array_equal(qs[i], qg[i]) and np.array_equal(d[i], dg[i]), (i, name)
        if expect is not None:
            assert bool(general[i]) == expect, (i, name)
