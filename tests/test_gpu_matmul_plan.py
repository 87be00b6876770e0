"""GPU parity of the prompt matmul at the sizes where its plan changes kernel (on long rows by 64 x 32 tiles per CU of a
256-CU GPU, below 128 tokens by the number of 64 x 16 tiles), with ragged rows, tokens and columns, against the decode GEMV of each token, bit for bit."""
import numpy as np
import pytest

from conftest import bits, load_synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [2, 3])
@pytest.mark.parametrize("rows,cols,n", [(2048, 2048, 256), (2048, 2048, 257), (2033, 2176, 270), (4096, 2048, 256),
                                         (4096, 2176, 257), (4100, 2304, 260), (4100, 2048, 130),
                                         (4864, 896, 33), (4864, 896, 49), (4850, 928, 77), (4864, 896, 127),
                                         (16384, 160, 17), (4096, 2080, 100), (4033, 4128, 97), (3072, 896, 64)])
def test_matmul_plan_boundaries_equal_gemv(qh, gpu, dtype, rows, cols, n):
    synth = load_synth()
    import torch
    host = synth.q8_tensor(rows + n, rows, cols) if dtype == 2 else synth.q4_tensor(rows + n, rows, cols, group=32)
    W = qh.DeviceTensor.upload(host, dtype, rows, cols)
    q, d = qh.quantize_q8(torch.from_numpy(synth.activations(cols, n, cols)).to(gpu))
    got = qh.matmul_q(W, q, d)
    for t in sorted({t for t in (0, 1, 15, 16, 31, 32, n // 2, n - 2, n - 1) if t < n}):
        want = qh.matvec_q(W, q[t], d[t])
        assert (bits(got[t].cpu().numpy()) == bits(want.cpu().numpy())).all(), t
