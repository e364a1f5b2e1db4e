"""The Python side of the file writers, on the CPU: the buffer it hands to the
C entry points, how often it calls them and what it returns."""
import ctypes
import sys

import pytest

from symphas_amd import abi, solver


class Writer:
    """A C entry point whose file has another text at each call (the field is
    advanced in between)."""

    def __init__(self, texts):
        self.texts = list(texts)
        self.calls = 0

    def __call__(self, buf, cap, n):
        self.calls += 1
        text = self.texts.pop(0) if len(self.texts) > 1 else self.texts[0]
        if buf is not None:
            if cap < len(text):
                return abi.E_INVALID
            ctypes.memmove(buf, text, len(text))
            if cap > len(text):
                ctypes.memset(buf.value + len(text), 0, 1)
        ctypes.cast(n, ctypes.POINTER(ctypes.c_size_t))[0] = len(text)
        return abi.OK


TEXTS = [
    [b"1.0 -2.0 3.0\n"],
    [b"1.0 -2.0 3.0\n", b"1.0 2.0 3.0\n"],              # shorter by the time it is written
    [b"1.0 2.0\n", b"-1.0 -2.0\n", b"-1.0 -2.0\n"],      # longer
    [b"1 2\n", b"-1 2\n", b"-1 2\n", b"-1 -2\n", b"-1 -2\n", b"1 -2\n"],
]


@pytest.mark.parametrize("texts", TEXTS)
def test_length_asked_for_first(texts):
    assert solver._file_bytes(Writer(texts)) == texts[-1]


@pytest.mark.parametrize("size", [5, 6, 40, 1000, 5_000_000])
def test_a_bound_takes_one_call(size):
    # every value is formatted in each call: with a bound there is one
    text = bytes(range(65, 91)) * (size // 26) + b"x" * (size % 26)
    for cap in (size, size + 1, size + 4096, 2 * size):
        w = Writer([text])
        out = solver._file_bytes(w, cap)
        assert w.calls == 1
        assert type(out) is bytes and out == text and hash(out) == hash(text)
        assert sys.getrefcount(out) == 2


def test_a_bound_that_is_too_small():
    # positions wider than the bound allows for
    w = Writer([b"123456789012345678.00 1.0\n"])
    assert solver._file_bytes(w, 10) == b"123456789012345678.00 1.0\n"
    assert w.calls == 3


def test_an_error_is_raised():
    w = Writer([b"1.0\n"])

    def call(buf, cap, n):
        return w(buf, cap, n) if buf is None else abi.E_HIP

    for cap in (0, 100):
        with pytest.raises(abi.SpsError) as e:
            solver._file_bytes(call, cap)
        assert e.value.status == abi.E_HIP
