"""GPU parity: prefill attention at the edges of its workgroups: chunks ending
before, at and after a workgroup's 256 (128) (token, head) columns and a 64-key
tile, sequences ending inside one, keys past a 1024-token page-entry span, the
tile widths' padding, and the last and first batch of the two workgroup orders
(31, 32 and 40 (sequence, KV head) pairs). Tolerance as for the other prefill
attention tests (2e-3 + 2e-2 |ref|).
"""
import pytest

pytest.importorskip("torch")

from tests.test_gpu_prefill_attention import check, run_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("past,new,Hq,Hkv,D,kw", [
    ([0, 63, 64, 0], [64, 65, 1, 129], 8, 2, 64, {}),            # G 4: 64 tokens a workgroup
    ([0, 1, 62], [31, 33, 32], 8, 2, 64, dict(fp8=True)),        # fp8, width 64: 32 tokens a workgroup
    ([1022, 960, 0], [3, 65, 70], 8, 2, 128, {}),                # across the span of 64 16-token pages
    ([2047, 10], [2, 5], 4, 4, 128, dict(fp8=True, P=32)),
    ([5, 0], [40, 85], 3, 1, 40, dict(paged=False)),             # G 3: 30 of 32 columns; rows padded to 64
    ([0, 100], [85, 86], 12, 4, 96, {}),                         # padded to 128
    ([0, 30], [34, 100], 16, 1, 32, dict(paged=False)),          # width 32, G 16: 2 tokens a wave
    ([3] * 31, [9] * 31, 4, 1, 64, {}),                          # 31 pairs: dealt over the XCDs
    ([3] * 16, [70, 9] * 8, 4, 2, 64, {}),                       # 32 pairs: an XCD each
    ([0] * 8, [65, 1, 2, 3, 4, 5, 6, 130], 5, 5, 64, {}),        # 40 pairs, G 1
])
def test_prefill_workgroup_edges(past, new, Hq, Hkv, D, kw):
    check(*run_prefill(past, new, Hq=Hq, Hkv=Hkv, D=D, seed=D + len(past), **kw))
