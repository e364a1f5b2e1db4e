"""The Python side of the file writers, on the CPU: the buffer it hands to the
C entry points and the length it returns."""
import ctypes

import pytest

from symphas_amd import abi, solver


class Writer:
    """A C entry point whose file has another text at each call (the field is
    advanced in between)."""

    def __init__(self, texts):
        self.texts = list(texts)

    def __call__(self, buf, cap, n):
        text = self.texts.pop(0) if len(self.texts) > 1 else self.texts[0]
        if buf is not None:
            if cap < len(text):
                return abi.E_INVALID
            ctypes.memmove(buf, text, len(text))
        ctypes.cast(n, ctypes.POINTER(ctypes.c_size_t))[0] = len(text)
        return abi.OK


@pytest.mark.parametrize("texts", [
    [b"1.0 -2.0 3.0\n"],
    [b"1.0 -2.0 3.0\n", b"1.0 2.0 3.0\n"],              # shorter by the time it is written
    [b"1.0 2.0\n", b"-1.0 -2.0\n", b"-1.0 -2.0\n"],      # longer
    [b"1 2\n", b"-1 2\n", b"-1 2\n", b"-1 -2\n", b"-1 -2\n", b"1 -2\n"],
])
def test_length_of_the_text_written(texts):
    assert solver._file_bytes(Writer(texts)) == texts[-1]


def test_an_error_is_raised():
    w = Writer([b"1.0\n"])

    def call(buf, cap, n):
        return w(buf, cap, n) if buf is None else abi.E_HIP

    with pytest.raises(abi.SpsError):
        solver._file_bytes(call)
