"""Argument checks of the entry points that take scratch (before any HIP call)."""

from __future__ import annotations

import ctypes

FAKE = 0x1000


def test_wide_entry_points_reject():
    from fused_decode import _lib as L

    lib = L.lib()

    def lin(m=32, n=64, k=128, sxm=128, swn=128, x=FAKE, w=FAKE, bias=None, bias_dtype=0, act=0):
        return lib.fd_linear_fp8_wide(FAKE, x, w, FAKE, bias, bias_dtype, None, 0, m, n, k, sxm, swn, 0, 0, 0, n, 1,
                                      None, 0, act, None)

    assert lin(act=2) == L.FD_EINVAL and lin(k=0) == L.FD_EINVAL and lin(m=-1) == L.FD_EINVAL
    assert lin(sxm=-8) == L.FD_EINVAL and lin(x=None) == L.FD_EINVAL and lin(bias=FAKE, bias_dtype=1) == L.FD_EINVAL
    assert lin(k=120) == L.FD_EUNSUPPORTED and lin(sxm=132) == L.FD_EUNSUPPORTED
    assert lin(swn=136) == L.FD_EUNSUPPORTED and lin(w=FAKE + 8) == L.FD_EUNSUPPORTED
    assert lin(m=0) == L.FD_OK and lin(n=0) == L.FD_OK
    gate = lambda m=32, h=128, i=64, x=FAKE, act=0: lib.fd_gate_up_fp8_wide(FAKE, x, FAKE, FAKE, m, h, i, h, act, None)
    assert gate(act=5) == L.FD_EINVAL and gate(h=0) == L.FD_EINVAL and gate(i=0) == L.FD_EINVAL
    assert gate(x=None) == L.FD_EINVAL and gate(h=120) == L.FD_EUNSUPPORTED and gate(m=0) == L.FD_OK


def test_wide_sizes_end_below_the_index_range():
    """The kernel's 32-bit indexes reach the end of the last tile, up to 127 rows past M and N."""
    from fused_decode import _lib as L

    lib, top = L.lib(), 2**31 - 1
    refused = lambda status: status == L.FD_EUNSUPPORTED and b"too large" in lib.fd_last_error()

    def lin(m, n):
        return lib.fd_linear_fp8_wide(FAKE, FAKE, FAKE, FAKE, None, 0, None, 0, m, n, 128, 128, 128, 0, 0, 0, n, 1, None,
                                      0, 0, None)

    for past in (top - 127, top - 15, top, top + 1):
        assert refused(lin(32, past)) and refused(lin(past, 64))
    half = (top + 1) // 2  # gate/up: 2 I weight rows
    for i in (half - 63, half):
        assert refused(lib.fd_gate_up_fp8_wide(FAKE, FAKE, FAKE, FAKE, 32, 128, i, 128, 0, None))


def test_wide_output_overlaps_no_operand():
    """Tiles are stored while other workgroups read: only row_add, element for element, may be the output."""
    from fused_decode import _lib as L

    lib, m, n, k = L.lib(), 32, 64, 128
    at = lambda i: 0x1000 + i * 0x100000
    y, x, w, s, b, r = (at(i) for i in range(6))
    over = lambda status: status == L.FD_EUNSUPPORTED and b"overlap" in lib.fd_last_error()

    def lin(y=y, x=x, w=w, s=s, b=b, r=r, bdt=L.FD_F32, rdt=L.FD_F16, srm=n, srn=1):
        return lib.fd_linear_fp8_wide(y, x, w, s, b, bdt, r, rdt, m, n, k, k, k, 1, srm, srn, n, 1, None, 0, L.FD_F16,
                                      None)

    last = m * n * 2 - 16  # bytes from the output's start to its last 16
    for arg in ({"x": y}, {"x": y + last}, {"w": y + last}, {"s": y + last}, {"b": y}, {"r": y, "srm": 0},
                {"r": y, "srm": 0, "srn": 0}, {"r": y + 16}, {"r": y, "srm": 1, "srn": m}, {"r": y, "rdt": L.FD_F32},
                {"r": y, "rdt": L.FD_BF16}, {"y": x + (m * k - 1) * 2}, {"y": w + n * k - 16}, {"y": s + n * 4 - 16}):
        assert over(lin(**arg)), arg
    i = k
    for arg in ((x, x, w, s), (w, x, w, s), (s, x, w, s), (x + (m * k - 8) * 2, x, w, s)):
        assert lib.fd_gate_up_fp8_wide(*arg, m, k, i, k, 0, None) == L.FD_EINVAL


def test_wide_scratch_follows_the_tiles():
    """No split, so no scratch, once the output tiles cover the GPU; else float32 sums for each split."""
    from fused_decode import _lib as L

    out = ctypes.c_int64(-1)
    ask = lambda m, n, k: (L.lib().fd_linear_fp8_wide_scratch(m, n, k, ctypes.byref(out)), out.value)
    assert ask(0, 64, 64) == (L.FD_OK, 0) and ask(32, 128, 256) == (L.FD_OK, 0)
    assert ask(300, 28672, 4096) == (L.FD_OK, 0)
    rc, got = ask(100, 4096, 14336)
    assert rc == L.FD_OK and got > 0 and got % (100 * 4096 * 4) == 0
    assert L.lib().fd_linear_fp8_wide_scratch(-1, 1, 1, ctypes.byref(out)) == L.FD_EINVAL


def test_kn_entry_points_reject():
    from fused_decode import _lib as L

    lib = L.lib()

    def lin(m=4, n=64, k=128, sxk=1, swk=64, x=FAKE, w=FAKE, bias=None, bias_dtype=0, act=0):
        return lib.fd_linear_kn(FAKE, x, w, bias, bias_dtype, None, 0, m, n, k, k, sxk, swk, 0, 0, 0, n, 1, None, 0,
                                act, None)

    assert lin(act=2) == L.FD_EINVAL and lin(k=0) == L.FD_EINVAL and lin(m=17) == L.FD_EINVAL
    assert lin(sxk=-1) == L.FD_EINVAL and lin(x=None) == L.FD_EINVAL and lin(bias=FAKE, bias_dtype=1) == L.FD_EINVAL
    assert lin(n=60) == L.FD_EUNSUPPORTED and lin(swk=68) == L.FD_EUNSUPPORTED
    assert lin(w=FAKE + 8) == L.FD_EUNSUPPORTED
    assert lin(m=0) == L.FD_OK and lin(n=0) == L.FD_OK
    out = ctypes.c_int64(-1)
    assert lib.fd_linear_kn_scratch(4, 4096, 4096, ctypes.byref(out)) == L.FD_OK
    assert out.value > 0 and out.value % (4 * 4096 * 4) == 0
    assert lib.fd_linear_kn_scratch(4, 65536, 4096, ctypes.byref(out)) == L.FD_OK and out.value == 0


def test_kn_output_overlaps_no_addend():
    """A column's rows are written by several threads: a bias or a broadcast row_add in the output is refused."""
    from fused_decode import _lib as L

    lib, m, n, k = L.lib(), 4, 64, 128
    y, x, w, b, r = (0x1000 + i * 0x100000 for i in range(5))

    def lin(b=b, r=r, bdt=L.FD_F32, rdt=L.FD_F16, srm=n, srn=1):
        return lib.fd_linear_kn(y, x, w, b, bdt, r, rdt, m, n, k, k, 1, n, 1, srm, srn, n, 1, None, 0, L.FD_F16, None)

    last = m * n * 2 - 16
    for arg in ({"b": y}, {"b": y + last}, {"r": y, "srm": 0}, {"r": y + last, "srm": 0}, {"r": y + 2},
                {"r": y, "srm": 1, "srn": m}, {"r": y, "rdt": L.FD_F32}):
        assert lin(**arg) == L.FD_EUNSUPPORTED and b"overlap" in lib.fd_last_error(), arg
