"""GPU parity of the prefill stack's attention (qh_attn.hip) where its launches change: rows on both sides of the one-launch
limit, pair groups that end in the middle, every head grouping, contexts that are no multiple of a cache block, a stack
larger than the score workspace, and values that overflow to infinity. The reference side is the same decoder at its
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


@pytest.mark.parametrize("turns", [(300,), (1500,)])
def test_stack_attention_infinite_values(qh, gpu, turns):
    """Value projections large enough that some rows overflow f16: an infinite value of a later token must not reach an
    earlier one (0 times it is NaN), so the second layer's cache rows stay equal."""
    qnt = qnt_module()
    hp = qnt.HParams(vocab_size=512, dim=256, n_layers=2, n_heads=4, n_kv_heads=1, head_dim=64, ffn_dim=512)
    tens = qnt.synthetic_q4mix(9, hp, shortlist=False)
    rec = tens["model.layers.0.self_attn.v_proj.weight"]
    data = np.array(rec.data)
    scales = data[rec.rows * rec.cols:].view(np.float16)
    scales[:] = (scales.astype(np.float32) * 3e5).astype(np.float16)  # |v| reaches 65,504 at a few positions
    tens["model.layers.0.self_attn.v_proj.weight"] = qnt.TensorRec(rec.dtype, rec.rows, rec.cols, data)
    _compare(qh, hp, tens, 1600, 512, turns)


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
