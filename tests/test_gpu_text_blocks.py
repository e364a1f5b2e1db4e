"""The checkpoint reader at the edges of its 4 KiB text blocks and the file
writers at the size where their buffers change."""
import numpy as np
import pytest

from symphas_amd import abi, models
from symphas_amd.solver import FDPlan

pytestmark = pytest.mark.gpu

SEPS = [" ", "\n", "  \t", "\r\n", "\v", "\f "]


@pytest.mark.parametrize("pad", [0, 1, 17, 4070, 4088, 4095, 4096, 4097, 8191])
def test_tokens_across_blocks(gpu_lib, pad):
    # tokens of 1 to 70 bytes (the longest and the odd ones go to the host's
    # parser) after `pad` spaces, so that they start, end and straddle anywhere
    rng = np.random.default_rng(pad)
    d = models.model_b((40, 30), dtype=abi.F64)
    tok, val = [], []
    for i in range(1200):
        v = rng.standard_normal() * 10.0 ** int(rng.integers(-5, 6))
        t = [f"{v:.10E}", f"{v:.3f}", f"{int(v)}", f"{v:.17e}", "0" * 50 + f"{abs(v):.6f}",
             "0" * 63 + str(int(rng.integers(0, 10))), "7"][int(rng.integers(0, 7))]
        tok.append(t)
        val.append(float(t))
    body = " " * pad + "".join(t + SEPS[int(rng.integers(0, len(SEPS)))] for t in tok)
    for text in (body, body + "1.5 2.5", body.rstrip()):
        with FDPlan(d) as p:
            idx = p.read_checkpoint(f"2 40 30 0.0 39.0 0.0 29.0 5 @{text}".encode())
            assert idx == 5
            assert np.array_equal(p.download().ravel(), np.array(val))


def test_large_files_equal_their_parts(gpu_lib):
    # above and below the size that asks for huge pages
    for n in ((64, 64), (640, 512)):
        d = models.model_b(n, dtype=abi.F32)
        psi = np.linspace(-1, 1, n[0] * n[1], dtype=np.float32).reshape(n[::-1])
        with FDPlan(d) as p:
            p.upload(psi)
            text = p.checkpoint_text(index=1)
            assert isinstance(text, bytes)
            assert text.split(b"@\n", 1)[1] == "".join(
                "".join("%.10E " % float(v) for v in row) + "\n" for row in psi).encode()
            assert np.array_equal(np.frombuffer(p.checkpoint_xdr()[-8 * psi.size:], ">f8"),
                                  psi.ravel().astype(np.float64))
            with FDPlan(d) as q:
                q.read_checkpoint(text)
                assert np.array_equal(q.download(), psi)
