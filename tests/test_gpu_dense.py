"""GPU parity of the unquantized matrices' kernels (qh_dense.hip) at the edges of their tiles: one token over 16-row and
64-row workgroups (row counts around both, the last tile of columns partial), and several tokens through the decoder's
32 x 32 tiles, against the oracle's serial chains, bit for bit."""
import numpy as np
import pytest

from conftest import bits, load_synth
from decoder_util import oracle_decoder, qnt_module
from test_gpu_decoder import _steps_vs_oracle

pytestmark = pytest.mark.gpu
F32, F16 = 0, 1


@pytest.mark.parametrize("dtype", [F32, F16])
@pytest.mark.parametrize("rows,cols", [(1, 32), (15, 64), (17, 224), (33, 288), (16, 4864), (200, 1056), (32767, 96),
                                       (32768, 32), (32833, 160)])
def test_matvec_ref_tiles_equal_oracle(qh, oracle, gpu, dtype, rows, cols):
    load_synth()
    import torch
    g = np.random.default_rng(rows + cols)
    w = (g.standard_normal((rows, cols)) * 0.02).astype(np.float16 if dtype == F16 else np.float32)
    x = g.standard_normal(cols).astype(np.float32)
    W = qh.DeviceTensor.upload(w.view(np.uint8).reshape(-1), dtype, rows, cols)
    got = qh.matvec_ref(W, torch.from_numpy(x).cuda()).cpu().numpy()
    want = oracle.matvec_f(dtype, rows, cols, w.view(np.uint8).reshape(-1), x)
    assert (bits(got) == bits(want)).all()


@pytest.mark.parametrize("dtype", [F32, F16])
@pytest.mark.parametrize("n", [2, 31, 33, 65])
def test_dense_prompt_equals_oracle(qh, oracle, gpu, dtype, n):
    """Prompts around the token tile (one launch of n tokens at a stack of 96), then decode steps."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=1000, dim=192, n_layers=2, n_heads=3, n_kv_heads=1, head_dim=64, ffn_dim=352)
    tens = qnt.synthetic_dense(60 + n, hp, dtype)
    orc = oracle_decoder(oracle, hp, tens, ctx_len=128)
    dec = qh.Decoder(hp, tens, ctx_len=128)
    dec.set_prefill_stack(96)
    ids = np.random.default_rng(n).integers(0, hp.vocab_size, n).astype(np.int32)
    _steps_vs_oracle(oracle, orc, dec, ids, 3, shortlist=False)
    dec.close()


@pytest.mark.parametrize("dtype", [F32, F16])
@pytest.mark.parametrize("rows,cols", [(8191, 416), (8193, 416), (16384, 192), (16385, 192), (16385, 224), (32769, 256),
                                       (32769, 288), (65536, 64), (65537, 64), (63, 32), (65, 64), (33, 96)])
def test_matvec_ref_forms_equal_oracle(qh, oracle, gpu, dtype, rows, cols):
    """Both sides of the lines between the one-token forms (16 or 64 rows to a workgroup, with or without loading
    waves)."""
    test_matvec_ref_tiles_equal_oracle(qh, oracle, gpu, dtype, rows, cols)


@pytest.mark.parametrize("dtype,ffn", [(F16, 4128), (F32, 8224)])
def test_merged_projections_in_many_rows_equal_oracle(qh, oracle, gpu, dtype, ffn):
    """Gate and up of one token in one launch of 64 rows to a workgroup (F16: 8,256 rows, with loading waves; F32: 16,448
    without), the second matrix beginning inside the grid."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=300, dim=64, n_layers=1, n_heads=1, n_kv_heads=1, head_dim=64, ffn_dim=ffn)
    tens = qnt.synthetic_dense(70, hp, dtype)
    orc = oracle_decoder(oracle, hp, tens, ctx_len=32)
    dec = qh.Decoder(hp, tens, ctx_len=32)
    ids = np.random.default_rng(4).integers(0, hp.vocab_size, 3).astype(np.int32)
    _steps_vs_oracle(oracle, orc, dec, ids, 3, shortlist=False)
    dec.close()
