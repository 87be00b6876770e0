"""quantize_q8 at the edges of its two kernels (16-byte lanes, and one element per lane for pointers that are not aligned
for them) against the oracle, byte for byte."""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,n", [(1, 32), (1, 96), (3, 32), (7, 896), (33, 1024), (5, 14336)])
@pytest.mark.parametrize("offset", [0, 1, 2])
def test_quantize_alignments(qh, oracle, gpu, n_tok, n, offset):
    import torch
    x = np.random.default_rng(n + n_tok).standard_normal((n_tok, n)).astype(np.float32)
    x[0, :32] = 0.0
    x[-1, -32:] *= 1e-35  # near the subnormals (below, 1 / scale overflows)
    buf = torch.zeros(n_tok * n + 4, device=gpu)
    xt = buf[offset:offset + n_tok * n].view(n_tok, n)
    xt.copy_(torch.from_numpy(x))
    q, d = qh.quantize_q8(xt)
    wq, wd = oracle.quantize_q8(x)
    assert (q.cpu().numpy() == wq).all() and (bits(d.cpu().numpy()) == bits(wd)).all()
