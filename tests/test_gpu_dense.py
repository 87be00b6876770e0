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


def _equal(a, b):
    """Equal bit for bit, any NaN equal to any other."""
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    return bool(((bits(a) == bits(b)) | (np.isnan(a) & np.isnan(b))).all())


def _special(g, shape, dtype):
    """Weights over the type's whole range (f16 and f32 subnormals, products that overflow and sums that come back), and
    infinities and NaN in a few rows."""
    f16 = dtype == F16
    w = (g.standard_normal(shape) * 2.0 ** g.integers(-24 if f16 else -148, 15 if f16 else 60, shape)).astype(np.float32)
    w[::5] = g.standard_normal(w[::5].shape) * (6e-8 if f16 else 1e-41)
    w[3::11, 7] = np.inf
    w[4::11, 40], w[4::11, 41] = np.inf, -np.inf
    w[6::11, 50] = np.nan
    with np.errstate(over="ignore"):
        return w.astype(np.float16 if f16 else np.float32)


@pytest.mark.parametrize("dtype", [F32, F16])
@pytest.mark.parametrize("rows,cols", [(70, 288), (8200, 416), (16400, 64)])
def test_matvec_ref_special_values_equal_oracle(qh, oracle, gpu, dtype, rows, cols):
    """The one-token forms on subnormal, overflowing, infinite and NaN weights and on such activations."""
    import torch
    load_synth()
    g = np.random.default_rng(rows)
    w = _special(g, (rows, cols), dtype).view(np.uint8).reshape(-1)
    W = qh.DeviceTensor.upload(w, dtype, rows, cols)
    for at, v in ((None, 0.0), (9, np.inf), (33, np.nan)):
        x = (g.standard_normal(cols) * 2.0 ** g.integers(-60, 40, cols)).astype(np.float32)
        x[::6] = 1e-40
        if at is not None:
            x[at] = v
        got = qh.matvec_ref(W, torch.from_numpy(x).cuda()).cpu().numpy()
        want = oracle.matvec_f(dtype, rows, cols, w, x)
        assert _equal(got, want) and (at or np.isfinite(want).mean() > 0.5)


@pytest.mark.parametrize("dtype", [F32, F16])
@pytest.mark.parametrize("n", [2, 33, 70])
def test_dense_prompt_special_values_equal_oracle(qh, oracle, gpu, dtype, n):
    """Several tokens through the f32 matrix instructions, against the oracle's multiply-add chains: tiny gate and wide up
    weights in the first layer; weights over the type's whole range, infinities and NaN in the last layer's k and v. Each
    k step is one fused multiply-add, rounded once, subnormals kept: every cache row of both layers, the hidden state and
    the logits are equal, and most of the last layer's values are finite."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=256, dim=128, n_layers=2, n_heads=2, n_kv_heads=1, head_dim=64, ffn_dim=352)
    tens = qnt.synthetic_dense(90 + n, hp, dtype)
    g = np.random.default_rng(n)

    def put(name, w):
        t = tens[name]
        tens[name] = qnt.TensorRec(t.dtype, t.rows, t.cols, np.ascontiguousarray(w).view(np.uint8).reshape(-1), t.ndim)

    # the last layer's k and v rows: stored in the cache as they come out, and read by the last token's output alone
    put("model.layers.1.self_attn.v_proj.weight", _special(g, (64, 128), dtype))
    put("model.layers.1.self_attn.k_proj.weight", _special(g, (64, 128), dtype))
    tiny = (g.standard_normal((352, 128)) * 2.0 ** g.integers(-24 if dtype == F16 else -140, -4, (352, 128)))
    put("model.layers.0.mlp.gate_proj.weight", tiny.astype(np.float16 if dtype == F16 else np.float32))
    wide = (g.standard_normal((352, 128)) * 2.0 ** g.integers(-12, 12, (352, 128)))
    put("model.layers.0.mlp.up_proj.weight", wide.astype(np.float16 if dtype == F16 else np.float32))
    orc = oracle_decoder(oracle, hp, tens, ctx_len=96, kv_f32=True)
    dec = qh.Decoder(hp, tens, ctx_len=96, kv_f32=True)
    dec.set_prefill_stack(96)
    ids = g.integers(0, hp.vocab_size, n).astype(np.int32)
    r = orc.forward_batch(ids, 0, top_k=0)
    dec.prefill(ids, 0, top_k=0)
    for l in range(2):
        for a, b in zip(dec.kv(l, n), orc.kv(l, n, 64)):
            assert _equal(a, b), l
    assert np.isfinite(dec.kv(1, n)[1]).mean() > 0.5
    assert _equal(dec.hidden(), r["hidden"]) and _equal(dec.logits(), r["logits"])
    dec.close()
