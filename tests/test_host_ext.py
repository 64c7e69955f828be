"""The native host side of the plugin steps (csrc/host_ext.cpp) where it can be
driven without a device."""
import subprocess
import sys
import textwrap

import pytest

from sga_amd import build as B


def _run(body):
    """``body`` in a process of its own (what it binds must not reach the other
    tests, and a crash must end nothing but it), with the extension as ``host``."""
    head = f"""
        import ctypes as C, importlib.util, sys
        import torch
        spec = importlib.util.spec_from_file_location("_host", {B.HOST_EXT!r})
        host = importlib.util.module_from_spec(spec)
        spec.loader.exec_module(host)
        nop = C.CFUNCTYPE(C.c_int)(lambda: 0)
        addr = C.cast(nop, C.c_void_p).value
        """
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(head) + textwrap.dedent(body)],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), (r.returncode, r.stdout, r.stderr)


def test_an_error_while_the_norm_is_read_raises():
    """The read of the norm is where an earlier device error surfaces: it has to
    arrive as an exception in a thread that holds the interpreter again.  A meta
    tensor stands for the device whose read fails."""
    _run("""
        host.bind(object, addr, addr, addr, addr)
        try:
            host.norm(torch.empty(64, dtype=torch.uint8, device="meta"), 1, 1, 0)
            raise SystemExit("no error")
        except RuntimeError as e:
            assert "meta" in str(e), e
        print("done")
        """)


def test_an_iterator_of_records_is_left_for_the_general_route():
    """What is not a list or a tuple is walked once, by the general route: had the
    native walk used it up, that route would see a step without records."""
    _run("""
        host.bind(object, addr, addr, addr, addr)
        for call in (lambda r: host.commit(r, False, -1, 1.0, False, False, 1.0, 1.0, False, 0),
                     lambda r: host.commit_compact(r, {}, None, True, 1.0, False, 1.0, False, 0),
                     lambda r: host.norm_table(r, True)):
            records = iter([object(), object()])
            assert call(records) is False
            assert len(list(records)) == 2
        print("done")
        """)


def test_scalars_are_taken_in_every_form_that_float_takes():
    import numpy as np
    import torch
    from sga_amd import _lib as L
    for x in ("0.1", 0.1, np.float64(0.1), np.float32(0.1), torch.tensor(0.1), torch.tensor([0.1])):
        assert L.f32(x) == float(np.float32(0.1))


@pytest.mark.parametrize("replay", [False, True])
def test_segment_tables_take_and_refuse_what_struct_fields_do(monkeypatch, replay):
    """Text that holds a number (learning rates and eps of a configuration file), numpy
    scalars and one-element tensors are numbers; a fractional offset is no offset."""
    import numpy as np
    import torch
    from sga_amd import _lib as L
    from sga_amd.segments import ReplaySegment, SegmentTable
    monkeypatch.setattr(L, "call", lambda *a: None)
    monkeypatch.setattr(L, "stream", lambda: 0)
    kw = dict(segs=not replay, rsegs=replay)
    rows = [dict(start=0, n=np.int64(5), b1=np.float64(0.9), b2=torch.tensor(0.95, dtype=torch.float64),
                 eps="1e-8", wd="0.1"),
            dict(start=5, n=7, b1=0.9, b2=0.95, eps=1e-8, wd=0.1)]
    t = SegmentTable(rows, "cpu", **kw)
    row_type = ReplaySegment if replay else L.Segment
    a, b = (row_type * 2).from_buffer_copy(bytes((t.rsegs if replay else t.segs).numpy()))
    assert (a.start, a.n, b.start, b.n) == (0, 5, 5, 7)
    for name in [f[0] for f in row_type._fields_][2:]:
        assert getattr(a, name) == getattr(b, name), name
    t.refresh(["1e-3", torch.tensor(2e-3, dtype=torch.float64)], 3)
    assert t._lr.tolist() == [1e-3, 2e-3] and t._bc2[0] == t._bc2[1] == np.float32(1 - 0.95 ** 3)
    for key, value in (("start", 0.5), ("n", 7.0)):
        with pytest.raises(TypeError):
            SegmentTable([dict(rows[1], **{key: value})], "cpu", **kw)


def test_words_that_have_not_arrived():
    """The wait ends by itself, and says which it was."""
    _run("""
        t = torch.full((3,), -1, dtype=torch.int32)
        assert host.arrived(t) is None
        t[0], t[1] = 7, -2
        assert host.arrived(t) is None
        t[2] = 0
        assert host.arrived(t) == (7, 2 ** 32 - 2, 0)
        for bad in (torch.zeros(2), torch.zeros(4, dtype=torch.int32)[::2], 3):
            try:
                host.arrived(bad)
                raise SystemExit("no error")
            except TypeError:
                pass
        print("done")
        """)


def test_results_of_64_bits_arrive_in_one_piece():
    """Either half may have all bits set (the low one of the double 2^53 - 1); the whole is looked at."""
    _run("""
        import struct
        t = torch.full((3,), -1, dtype=torch.int64)
        assert host.arrived(t) is None
        low = struct.unpack("<q", struct.pack("<d", 2.0 ** 53 - 1))[0]
        t[0], t[1] = low, 7
        assert low & 0xFFFFFFFF == 0xFFFFFFFF and host.arrived(t) is None
        t[2] = -(1 << 32)
        assert host.arrived(t) == (low, 7, 2 ** 64 - 2 ** 32)
        assert host.arrived(t[:1]) == (low,)
        print("done")
        """)


def test_a_norm_that_no_kernel_has_written_raises():
    """The bound function here writes nothing: its word is no norm (read as a float it is NaN)."""
    _run("""
        host.bind(object, addr, addr, addr, addr)
        try:
            print(host.norm(torch.zeros(64, dtype=torch.uint8), 1, 1, 0))
        except RuntimeError as e:
            assert "not arrived" in str(e), e
            print("done")
        """)
