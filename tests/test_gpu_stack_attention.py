"""GPU parity of the prefill stack's attention (qh_attn.hip) where its launches change: rows on both sides of the one-launch
limit and of the sizes where the number of workgroups decides, pair groups that end in the middle, 1, 2, 3, 4 and 7 query
heads to a KV head, contexts that are no multiple of a cache block, a stack larger than the score workspace or with a
smaller one, and infinite values and keys. The reference side is the same decoder at its
default 32-token chunks (attention_kernel, itself compared with the oracle in test_gpu_decoder.py and test_gpu_options.py):
states, logits and every cache row must be equal bit for bit."""
import numpy as np
import pytest

from decoder_util import qnt_module

pytestmark = pytest.mark.gpu


def _equal(a, b):
    a, b = np.asarray(a), np.asarray(b)
    if a.dtype == np.uint16:  # f16 bits; a NaN's sign and payload are not pinned
        a, b = a.view(np.float16), b.view(np.float16)
    same = a.view(np.uint16 if a.itemsize == 2 else np.uint32) == b.view(np.uint16 if b.itemsize == 2 else np.uint32)
    return bool((same | (np.isnan(a) & np.isnan(b))).all())


def _compare(qh, hp, tens, ctx, stack, turns, seed=3):
    ids = np.random.default_rng(seed).integers(0, hp.vocab_size, sum(turns)).astype(np.int32)
    decs = []
    for s in (32, stack):
        dec = qh.Decoder(hp, tens, ctx_len=ctx)
        dec.set_prefill_stack(s)
        decs.append(dec)
    pos = 0
    for n in turns:
        for dec in decs:
            dec.prefill(ids[pos:pos + n], pos, top_k=0)
        assert _equal(decs[0].hidden(), decs[1].hidden()), f"hidden state after {pos + n} tokens"
        assert _equal(decs[0].logits(), decs[1].logits()), f"logits after {pos + n} tokens"
        pos += n
    for l in range(hp.n_layers):
        for a, b in zip(decs[0].kv(l, pos), decs[1].kv(l, pos)):
            assert _equal(a, b), f"layer {l} cache"
    for dec in decs:
        assert dec.status() == 0
        dec.close()


@pytest.mark.parametrize("n_heads,n_kv,head_dim,ctx,stack,turns", [
    (4, 1, 64, 1501, 1024, (1, 33, 990, 64, 300)),   # up to 1,024 rows in one launch, then the three
    (4, 4, 64, 1333, 544, (540, 700)),               # one query head per KV head: a group spans 64 tokens
    (14, 2, 64, 1203, 96, (40, 1000, 77)),           # 7 heads per KV head: groups end inside a token
    (2, 1, 128, 1451, 256, (129, 1200, 35)),
    (6, 2, 128, 1100, 1024, (17, 1080)),
])
def test_stack_attention_equals_chunks(qh, gpu, n_heads, n_kv, head_dim, ctx, stack, turns):
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=512, dim=n_heads * head_dim, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv,
                     head_dim=head_dim, ffn_dim=512)
    _compare(qh, hp, qnt.synthetic_q4mix(51 + n_heads, hp, shortlist=False), ctx, stack, turns)


def test_stack_attention_larger_than_its_workspace(qh, gpu):
    """1,024 tokens of 14 heads over 5,600 rows hold more scores than the workspace: several passes over the stack."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=512, n_layers=1, ffn_dim=512)
    _compare(qh, hp, qnt.synthetic_q4mix(7, hp, shortlist=False), 8192, 1024, (5600,))


_OUTLIER = 511  # the token whose rows overflow


def _outlier_model(qnt, kind):
    """A two-layer model in which one token, and no other, has an infinite value (kind "value": dimension 7) or key
    (dimension 31, which RoPE hardly turns at these positions): its embedding is 0 but for one dimension, which every
    other token has 0 in, and one projection row weighs that dimension with 5,080 (normed it is 16; f16 ends at 65,504).
    "key_low": every head's q is negative there, the score -inf; "key_high": positive, +inf; "key_nan": a second infinite
    dimension with the other sign, NaN."""
    hp = qnt.HParams(vocab_size=512, dim=256, n_layers=2, n_heads=4, n_kv_heads=1, head_dim=64, ffn_dim=512)
    tens = qnt.synthetic_q4mix(9, hp, shortlist=False)

    def edit(name):
        rec = tens[name]
        data = np.array(rec.data)
        tens[name] = qnt.TensorRec(rec.dtype, rec.rows, rec.cols, data, rec.ndim)
        return data[:rec.rows * rec.cols].view(np.int8).reshape(rec.rows, rec.cols), \
            data[rec.rows * rec.cols:].view(np.float16).reshape(rec.rows, rec.cols // 32)

    codes, scales = edit("model.embed_tokens.weight")
    codes[:, 5] = 0
    codes[_OUTLIER] = 0
    codes[_OUTLIER, 5], scales[_OUTLIER, 0] = 127, 0.02
    p = "model.layers.0.self_attn."
    codes, scales = edit(p + ("v" if kind == "value" else "k") + "_proj.weight")
    for r in (7,) if kind == "value" else (31,) if kind != "key_nan" else (31, 30):
        codes[r, :32], codes[r, 5], scales[r, 0] = 0, 127, 40.0
    if kind != "value":
        rec = tens[p + "q_proj.bias"]
        bias = np.array(rec.data).view(np.float32).copy()
        bias.reshape(4, 64)[:, 31] = -4.0 if kind == "key_low" else 4.0
        bias.reshape(4, 64)[:, 30] = -4.0
        tens[p + "q_proj.bias"] = qnt.TensorRec(rec.dtype, rec.rows, rec.cols, bias.view(np.uint8), rec.ndim)
    return hp, tens


@pytest.mark.parametrize("kind", ["value", "key_low", "key_high", "key_nan"])
@pytest.mark.parametrize("turns,at", [
    ((300,), (201, 202, 203, 255)),         # four tokens of a head to a workgroup
    ((900,), (801, 802, 803, 863)),         # 16 pairs (four tokens) to a workgroup
    ((900, 400), (1101, 1102, 1103, 1215)),  # 64 pairs (16 tokens) to a group, three launches
])
def test_stack_attention_infinite_values(qh, gpu, turns, at, kind):
    """One infinite value or key, at a position inside a workgroup's or group's tokens and inside a step of four rows, or
    the last row of a tile: it must not reach a token before it (0 times it is NaN), whose second-layer cache rows stay
    those of a prompt without it. A score of -inf has the weight 0, so that later tokens' rows stay finite too; after the
    others they are NaN. Equal to the 32-token chunks bit for bit."""
    qnt = qnt_module()
    hp, tens = _outlier_model(qnt, kind)
    n = sum(turns)
    plain = np.random.default_rng(3).integers(0, _OUTLIER, n).astype(np.int32)
    decs = []
    for stack in (32, 1024):
        dec = qh.Decoder(hp, tens, ctx_len=1408)
        dec.set_prefill_stack(stack)
        decs.append(dec)

    def run(dec, ids):
        pos = 0
        for m in turns:
            dec.prefill(ids[pos:pos + m], pos, top_k=0)
            pos += m
        return [c.view(np.float16) for l in range(2) for c in dec.kv(l, n)]

    base = run(decs[1], plain)
    assert all(np.isfinite(c).all() for c in base)
    for p in at:
        ids = plain.copy()
        ids[p] = _OUTLIER
        want, got = run(decs[0], ids), run(decs[1], ids)
        inf0 = ~np.isfinite(want[1] if kind == "value" else want[0])  # layer 0: infinite there and nowhere else
        assert inf0[p].any() and not np.delete(inf0, p, 0).any()
        for w, b in zip(want[2:], base[2:]):  # layer 1
            assert (w[:p] == b[:p]).all() and np.isfinite(w[:p]).all()
            assert np.isfinite(w[p:]).all() if kind == "key_low" else np.isnan(w[p:]).any(1).all()
        for w, g in zip(want, got):
            assert _equal(w.view(np.uint16), g.view(np.uint16)), p
    for dec in decs:
        dec.close()
    q = tens["model.layers.0.self_attn.q_proj.weight"]  # layer 1 does depend on layer 0's attention
    tens["model.layers.0.self_attn.q_proj.weight"] = qnt.TensorRec(q.dtype, q.rows, q.cols, np.zeros_like(q.data))
    dec = qh.Decoder(hp, tens, ctx_len=1408)
    dec.set_prefill_stack(1024)
    other = run(dec, plain)
    dec.close()
    assert (other[2][2:] != base[2][2:]).any(1).mean() > 0.99


@pytest.mark.parametrize("n_heads,n_kv,head_dim,ctx,stack,turns", [
    # up to 1,024 rows a workgroup takes four tokens of a head (up to 819 workgroups at position 0, 512 later on a
    # 256-CU GPU) or 16 pairs; past them a head and token (up to 512, or 1,024 on few rows) or pair groups
    (14, 2, 64, 1400, 256, (231, 145, 146, 236, 33, 36, 37, 73, 74, 200)),
    (4, 1, 64, 1800, 1024, (819, 64, 128, 129, 256, 257)),
    (6, 6, 64, 1450, 512, (35, 340, 420, 85, 200, 170, 171)),
    # head_dim 128: a head and token for one round of workgroups, or two past a mean of 200 rows, to 1,024 rows; one
    # round to 2,700
    (4, 2, 128, 1300, 256, (64, 65, 128, 129, 256, 128, 129, 63, 64, 65)),
    (2, 1, 128, 2900, 1024, (2600, 64, 64, 129)),
])
def test_small_stacks_equal_chunks(qh, gpu, n_heads, n_kv, head_dim, ctx, stack, turns):
    """Turns on both sides of the sizes where the stack's attention changes kernel by its number of workgroups."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=512, dim=n_heads * head_dim, n_layers=2, n_heads=n_heads, n_kv_heads=n_kv,
                     head_dim=head_dim, ffn_dim=512)
    _compare(qh, hp, qnt.synthetic_q4mix(83 + n_heads, hp, shortlist=False), ctx, stack, turns, seed=5)


def _wide(qnt):
    hp = qnt.HParams(vocab_size=512, dim=1024, n_layers=1, n_heads=16, n_kv_heads=2, head_dim=64, ffn_dim=512)
    return hp, qnt.synthetic_q4mix(17, hp, shortlist=False)


def test_stack_takes_no_score_workspace_for_a_short_context(qh, gpu):
    """A context of up to 1,024 rows never goes through the score workspace (69 MB for this model's 1,024-token stack):
    setting the stack takes its work buffers (about 20 MB) and no more."""
    import torch
    qnt = qnt_module()
    hp, tens = _wide(qnt)
    dec = qh.Decoder(hp, tens, ctx_len=1024)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    dec.set_prefill_stack(1024)
    taken = free - torch.cuda.mem_get_info()[0]
    dec.close()
    assert taken < 48 << 20, taken


def test_stack_with_a_smaller_score_workspace(qh, gpu):
    """Where the score workspace cannot be allocated whole the stack is still set, with half of it (here its allocation,
    the thirteenth, is made to fail), and its attention takes the stack in more passes with the same results."""
    qnt = qnt_module()
    hp, tens = _wide(qnt)
    ids = np.random.default_rng(9).integers(0, hp.vocab_size, 1800).astype(np.int32)
    got = []
    for after in (-1, 12):
        dec = qh.Decoder(hp, tens, ctx_len=1900)
        try:
            qh.lib().qh_fault_alloc(after)
            dec.set_prefill_stack(1024)
        finally:
            qh.lib().qh_fault_alloc(-1)
        dec.prefill(ids, 0, top_k=0)
        got.append((dec.hidden(), dec.kv(0, len(ids))))
        dec.close()
    assert _equal(got[0][0], got[1][0])
    assert all(_equal(a, b) for a, b in zip(got[0][1], got[1][1]))


@pytest.mark.parametrize("dtype", [2, 3])
def test_wide_model_stack_equals_chunks(qh, gpu, dtype):
    """Rows of 2,048 with more than two 64 x 32 tiles per CU: the prompt matmul's plan with 4-block chunks, which on a stack
    also takes gate and up with SwiGLU in the epilogue, in whole and ragged token tiles."""
    qnt = qnt_module()
    import quanta_cpp_amd.synth as synth
    hp = qnt.HParams(vocab_size=512, dim=2048, n_layers=1, n_heads=32, n_kv_heads=8, head_dim=64, ffn_dim=4352)
    tens = qnt.synthetic_q4mix(19, hp, shortlist=False)
    if dtype == 2:
        for i, (n, r, c) in enumerate((("gate", 4352, 2048), ("up", 4352, 2048), ("down", 2048, 4352))):
            tens["model.layers.0.mlp.%s_proj.weight" % n] = qnt.TensorRec(2, r, c, synth.q8_tensor(900 + i, r, c))
    _compare(qh, hp, tens, 320, 160, (160, 131))
