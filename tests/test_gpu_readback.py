"""Fields leave through pinned chunks (64 Ki values and up, 16 slots of 2 MiB):
what is written comes back, in one chunk, in several and after the slots wrap,
to arrays at any 8-byte alignment, from several threads."""

import ctypes
import threading

import numpy as np
import pytest

from xfdtd_core_amd import native

pytestmark = pytest.mark.gpu


def _context(n, dtype):
    ext = lambda c, e: tuple(m + (1 if (q != c if e else q == c) else 0) for q, m in enumerate(n))  # noqa: E731
    coeffs = {}
    for name in native.COEFF_NAMES:
        e = name[1] == "e"
        coeffs[name] = np.full(ext("xyz".index(name[2]), e), 0.5)
    return native.Context(coeffs, dtype)


@pytest.mark.parametrize("dtype", ["f64", "f32"])
@pytest.mark.parametrize("n", [(3, 4, 5), (31, 63, 31), (32, 63, 32), (130, 129, 131), (190, 170, 180)])
def test_read_returns_what_was_written(n, dtype):
    ctx, L = _context(n, dtype), native.load_library()
    rng = np.random.default_rng(n[0])
    ext = (n[0], n[1] + 1, n[2] + 1)
    v = rng.standard_normal(ext)
    want = v.astype(np.float32).astype(np.float64) if dtype == "f32" else v
    ctx.write("EX", v)
    np.testing.assert_array_equal(ctx.read("EX"), want)
    room = np.full(v.size + 3, -1.0)  # an odd place in a larger array
    assert L.xfd_read_field(ctx._h, 0, ctypes.c_void_p(room[1:].ctypes.data)) == 0
    np.testing.assert_array_equal(room[1:-2].reshape(ext), want)
    assert room[0] == room[-1] == room[-2] == -1.0


# four reads run at a time; more wait, and small reads do beside large ones
@pytest.mark.parametrize("sizes", [[(90, 80, 70)] * 3, [(90, 80, 70), (5, 6, 7), (64, 64, 64)] * 3,
                                   [(150, 140, 130)] * 2 + [(9, 9, 9)] * 6])
def test_reads_from_several_threads(sizes):
    jobs = []
    for q, n in enumerate(sizes):
        ctx = _context(n, "f64")
        v = np.random.default_rng(q).standard_normal((n[0], n[1] + 1, n[2] + 1))
        ctx.write("EX", v)
        jobs.append((ctx, v, []))
    threads = [threading.Thread(target=lambda j=j: j[2].extend(j[0].read("EX") for _ in range(4))) for j in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for _, v, got in jobs:
        assert len(got) == 4
        for g in got:
            np.testing.assert_array_equal(g, v)
