"""GPU parity: merging the balanced partition's pieces, at the edges of the
dispatch between the wide merge (few (sequence, KV head) segments of many
tiles) and the one-wave merge, and of the wide merge's own splits: one piece, fewer pieces
than its four waves, one past a wave's 16-row batch, more than 64 pieces a wave
(a lane each), sequences with nothing cached, every tile width and group size;
NaN and infinite scores on both sides of the dispatch.

Tolerance: the decode attention tests' (2e-3 + 2e-2 |ref|): the merge is the
same fp32 sum of the same pieces in another order.
"""
import pytest

torch = pytest.importorskip("torch")

from tests.kv_inputs import sm_scale
from tests.test_gpu_decode_attention import assert_close, run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,Hq,Hkv,D,kw", [
    ([1], 4, 1, 128, {}),                                   # one piece
    ([70], 16, 1, 64, {}),                                  # three tiles: a wave without a piece, G 16
    ([65 * 32 + 1], 8, 2, 128, {}),                         # 66 pieces: 17 in a wave
    ([9000], 4, 1, 128, dict(paged=True)),                  # 282 one-tile pieces: more than 64 in a wave
    ([33000], 3, 1, 64, {}),                                # W >= NW: every wave holds a piece, G 3
    ([8000, 1, 300], 10, 2, 32, {}),                        # 32-wide rows, G 5
    ([700, 33, 1200], 8, 4, 96, dict(fp8=True, paged=True)),
    ([40] * 32, 16, 8, 64, dict(zero_first=True)),          # 256 short segments: the one-wave merge
    ([40] * 33, 16, 8, 64, dict(zero_first=True)),          # 264: always that one
    ([65] * 32, 8, 8, 64, {}),                              # G 1: three tiles take the wide merge,
    ([64] * 4, 8, 8, 64, {}),                               # two the one-wave merge
    ([64] * 17, 24, 8, 64, {}),                             # 136 segments, G 3: the wide at up to two tiles,
    ([128] * 17, 24, 8, 64, {}),                            # the one-wave merge at three and four,
    ([129] * 24, 24, 8, 64, {}),                            # the wide again from five on
    ([64] * 17, 16, 8, 64, {}),                             # G 2: the one-wave merge at up to two tiles,
    ([65] * 24, 16, 8, 128, {}),                            # the wide from three on
    ([384] * 32, 16, 8, 64, {}),                            # 256: up to twelve tiles the one-wave merge,
    ([385] * 32, 16, 8, 64, {}),                            # thirteen the wide, except
    ([385] * 32, 16, 8, 128, {}),                           # on 128-wide tiles
])
def test_merge_edges(lengths, Hq, Hkv, D, kw):
    got, ref, _ = run_case(lengths, Hq=Hq, Hkv=Hkv, D=D, seed=len(lengths) + D, **kw)
    if kw.get("zero_first"):
        assert (got[0] == 0).all()
        got, ref = got[1:], ref[1:]
    assert_close(got, ref)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("batch", [16, 32, 33])  # 128 segments: the wide merge; 264: the one-wave; 256: by length
@pytest.mark.parametrize("lengths", [40, 700])
def test_nan_and_infinite_scores_stay(D, batch, lengths):
    # A NaN in q, a NaN in a cached key, an infinite score: NaN rows as softmax gives them, not zeros; a score
    # of -inf drops its key. Every other row is as close as ever.
    from tinytron_amd import ops

    g = torch.Generator(device="cuda").manual_seed(D + batch)
    Hkv, G, cap = 8, 2, 704
    q = torch.randn(batch, Hkv * G, D, generator=g, device="cuda").bfloat16()
    k, v = (torch.randn(batch, Hkv, cap, D, generator=g, device="cuda").bfloat16() for _ in "kv")
    q[1, 3, D - 1] = float("nan")
    k[2, 4, lengths // 2, 0] = float("nan")
    k[3, 5, lengths // 2, 1] = float("inf")  # +inf or -inf by the sign of each head's q[1]
    q[3, 10, 1], q[3, 11, 1] = 1.0, -1.0
    kv = ops.KVLayout(k=k.view(-1), v=v.view(-1), strides=(Hkv * cap * D, 16 * D, cap * D), num_heads=Hkv, head_dim=D,
                      page_size=16, capacity=cap, kind="bf16")
    lens = torch.full((batch,), lengths, dtype=torch.int32, device="cuda")
    got = ops.decode_attention(q, kv, lens, lengths).float().cpu()
    kc, vc = (x[:, :, :lengths].float().cpu().repeat_interleave(G, dim=1) for x in (k, v))
    scores = (q.float().cpu()[:, :, None] * kc).sum(-1) * sm_scale(D)
    ref = (torch.softmax(scores, -1)[..., None] * vc).sum(2)
    nan = torch.isnan(ref)
    assert nan[1, 3].all() and nan[2, 8:10].all() and nan[3, 10].all() and not nan[3, 11].any() and nan.sum() == 4 * D
    assert torch.equal(torch.isnan(got), nan)
    assert_close(got[~nan].numpy(), ref[~nan].numpy())
