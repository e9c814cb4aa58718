"""GPU parity: merging the balanced partition's pieces, at the edges of the
dispatch between the wide merge (at most 256 (sequence, KV head) segments) and
the one-wave merge, and of the wide merge's own splits: one piece, fewer pieces
than its four waves, one past a wave's 16-row batch, more than 64 pieces a wave
(a lane each), sequences with nothing cached, every tile width and group size.

Tolerance: the decode attention tests' (2e-3 + 2e-2 |ref|): the merge is the
same fp32 sum of the same pieces in another order.
"""
import pytest

torch = pytest.importorskip("torch")

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
    ([40] * 32, 16, 8, 64, dict(zero_first=True)),          # 256 segments: the last the wide merge takes
    ([40] * 33, 16, 8, 64, dict(zero_first=True)),          # 264: the one-wave merge
])
def test_merge_edges(lengths, Hq, Hkv, D, kw):
    got, ref, _ = run_case(lengths, Hq=Hq, Hkv=Hkv, D=D, seed=len(lengths) + D, **kw)
    if kw.get("zero_first"):
        assert (got[0] == 0).all()
        got, ref = got[1:], ref[1:]
    assert_close(got, ref)
