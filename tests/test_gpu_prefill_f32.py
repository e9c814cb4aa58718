"""GPU parity: fp32 prefill attention (tt_prefill_attn_f32) vs the fp64 oracle
and vs row attention, at the edges of its tiles: head dims filling and padding
each tile width, chunks that end inside, at and after a 32-key tile and a
wave's turn, one and two column blocks per workgroup, group sizes that leave
columns idle, rows past new_lens (zeros), NaN in every unused slot.

Tolerance as for the row attention tests' fp32 caches: 1e-5 + 1e-4 |ref| (fp32
operands and sums of up to 1300 terms in another order).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle.attention import prefill_attention as ref_prefill
from tests.kv_inputs import sm_scale
from tests.test_gpu_rows_attention import _cache, _dev, _queries

pytestmark = pytest.mark.gpu


def _run(cached, new, Hq, Hkv, D, paged, seed=0, T=None, edit=None):
    from tinytron_amd import ops

    rng = np.random.default_rng(seed)
    T = T or max(new)
    kv, keys, values = _cache([c + n for c, n in zip(cached, new)], Hkv, D, "f32", paged, rng)
    if edit is not None:
        edit(kv, values)
    q, qf = _queries(rng, (len(cached), Hq, T, D), "f32")
    assert ops.prefill_f32_supported(kv, Hq)
    pos = torch.tensor(cached, dtype=torch.int32, device="cuda")
    nl = torch.tensor(new, dtype=torch.int32, device="cuda")
    out = torch.full((len(cached), T, Hq, D), float("nan"), device="cuda")
    ops.prefill_attention_f32(q, kv, pos, max(c + n for c, n in zip(cached, new)), new_lens=nl, out=out)
    torch.cuda.synchronize()
    ref = ref_prefill(qf, keys, values, cached, new, Hkv, sm_scale(D))
    return out.cpu().numpy(), ref, (ops, q, kv)


def _check(got, ref, new):
    for b, n in enumerate(new):
        assert np.all(got[b, n:] == 0.0)
        err = np.abs(got[b, :n] - ref[b][:n])
        assert np.all(err <= 1e-5 + 1e-4 * np.abs(ref[b][:n])), (b, float(err.max()))


@pytest.mark.parametrize("D", [4, 20, 32, 36, 64, 96, 128])
@pytest.mark.parametrize("paged", [False, True])
def test_head_dims(D, paged):
    cached, new = [0, 40, 5, 127, 0], [33, 1, 17, 66, 0]
    got, ref, _ = _run(cached, new, 6, 2, D, paged, seed=D)
    _check(got, ref, new)


@pytest.mark.parametrize("Hq,Hkv", [(4, 4), (5, 1), (16, 1), (16, 8)])
def test_groups_and_long_prefix(Hq, Hkv):
    # past one 1024-token page-entry span; keys at 31, 32, 33 and 127 .. 129
    cached, new = [1250, 30, 0], [37, 3, 129]
    got, ref, _ = _run(cached, new, Hq, Hkv, 64, True, seed=Hq)
    _check(got, ref, new)


def test_two_blocks_per_workgroup():
    # 8 sequences x 8 heads x 130 / 8 token blocks: past two workgroups per CU
    cached, new = [0, 3, 64, 0, 1, 0, 31, 2], [130, 64, 9, 17, 130, 1, 100, 16]
    got, ref, (ops, q, kv) = _run(cached, new, 32, 8, 32, False, seed=9)
    _check(got, ref, new)
    rows = ops.prefill_attention_rows(q, kv, cached, new)
    assert torch.allclose(torch.from_numpy(got), rows.cpu(), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("Hq,Hkv,D,paged,batch,cached", [
    (4, 1, 64, False, 1, 0),
    (4, 1, 128, False, 1, 0),      # width 128
    (3, 1, 100, True, 2, 37),      # padded to 128, page pool, a prefix
    (2, 2, 20, True, 1, 5),        # padded to 32, G 1: sixteen tokens a block
    (32, 8, 32, False, 8, 0),      # two column blocks per workgroup
    (32, 8, 64, True, 8, 3),
])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_non_finite_value_of_a_later_token_stays_there(Hq, Hkv, D, paged, batch, cached, value):
    # value row `token` of each chunk is inf or NaN: it and later tokens see it, earlier ones (same tile, same
    # block of columns) must not
    new = 136 if batch == 8 else 40
    token = new - 20

    def edit(kv, values):
        v = kv.v.view(-1)
        for b in range(batch):
            t = cached + token
            if paged:
                page = int(kv.page_table[b, t // kv.page_size])
                row = page * kv.strides[1] + t % kv.page_size * D
            else:
                row = b * kv.strides[0] + t * D
            for h in range(Hkv):
                v[row + h * kv.strides[2]:][:D] = value

    got, ref, _ = _run([cached] * batch, [new] * batch, Hq, Hkv, D, paged, seed=3, edit=edit)
    _check(got[:, :token], [r[:token] for r in ref], [token] * batch)
    later = got[:, token:]
    assert np.all(np.isinf(later) if np.isinf(value) else np.isnan(later))


def _layer(B, Hkv, D, cap, seed):
    from tinytron_amd.cache import LayerPagedKVCache

    c = LayerPagedKVCache(B, Hkv, D, cap, 16, "cuda", torch.float32)
    g = torch.Generator(device="cuda").manual_seed(seed)
    c.layout.k.normal_(generator=g)
    c.layout.v.normal_(generator=g)
    return c, g


def test_chunk_after_set_lengths_and_over_two_appends():
    # The chunk ends at each sequence's length as the cache knows it, however the tokens came there.
    from tinytron_amd import ops

    B, Hq, Hkv, D, T = 2, 4, 2, 64, 6
    c, g = _layer(B, Hkv, D, 64, 5)
    q = torch.randn(B, Hq, T, D, generator=g, device="cuda")
    c.set_lengths([40, 23])
    got = c.prefill_attend(q, [6, 4])
    assert torch.allclose(got, c.prefill_attend(q, [6, 4], kernel=False), rtol=1e-4, atol=1e-5)
    table = ops.build_rope_table(64, D, dtype=torch.float32, device="cuda")
    k = torch.randn(B, Hkv, 3, D, generator=g, device="cuda")
    rot = torch.cat([c.rope_append(q[:, :, i:i + 3], k, k, table) for i in (0, 3)], dim=2)
    assert c.seq_lens_host == [46, 29]
    got = c.prefill_attend(rot, [6, 6])
    assert torch.allclose(got, c.prefill_attend(rot, [6, 6], kernel=False), rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("form", ["q_strided", "q_token_major", "out_strided", "out_rows", "out_bf16"])
def test_forms_that_row_attention_took(form):
    # views of q and out that the kernel reads or writes directly, and those that go on taking row attention
    B, Hq, Hkv, D, T = 2, 4, 2, 32, 7
    c, g = _layer(B, Hkv, D, 48, 6)
    c.set_lengths([40, 23])
    q = torch.randn(B, Hq, T, D, generator=g, device="cuda")
    ref = c.prefill_attend(q, [7, 4], kernel=False)
    out = None
    if form == "q_strided":
        q = torch.stack([q, q + 1], -1)[..., 0]
    elif form == "q_token_major":
        q = q.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "out_strided":
        out = torch.empty(B, T, Hq, D, 2, device="cuda")[..., 1]
    elif form == "out_rows":
        out = torch.empty(B * T, Hq * D, device="cuda")
    else:
        out = torch.empty(B, T, D, Hq, device="cuda", dtype=torch.bfloat16).transpose(2, 3)
    got = c.prefill_attend(q, [7, 4], out=out)
    assert out is None or got is out
    tol = dict(rtol=2.0 ** -8, atol=1e-5) if form == "out_bf16" else dict(rtol=1e-4, atol=1e-5)
    assert torch.allclose(got.float().reshape(ref.shape), ref, **tol)


def test_out_that_does_not_fit_is_refused():
    from tinytron_amd import ops

    c, g = _layer(2, 2, 32, 48, 7)
    c.set_lengths([40, 23])
    q = torch.randn(2, 4, 7, 32, generator=g, device="cuda")
    pos = torch.tensor([33, 16], dtype=torch.int32, device="cuda")
    for shape, dtype in [((2, 6, 4, 32), torch.float32), ((2, 7, 4, 32), torch.bfloat16), ((2, 7, 4, 36), torch.float32)]:
        out = torch.empty(shape, dtype=dtype, device="cuda")
        with pytest.raises(ValueError, match="out"):
            ops.prefill_attention_f32(q, c.layout, pos, 40, out=out)
    with pytest.raises(RuntimeError):
        c.prefill_attend(q, [7, 7], out=torch.empty(2, 6, 4, 32, device="cuda"))
    for where in (dict(out=torch.empty(2, 7, 4, 32)), dict(new_lens=torch.tensor([7, 7], dtype=torch.int32))):
        with pytest.raises(ValueError):
            ops.prefill_attention_f32(q, c.layout, pos, 40, **where)
