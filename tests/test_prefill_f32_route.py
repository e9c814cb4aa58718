"""Which route an fp32 prompt chunk takes: the fp32 prefill kernel, or row
attention for a few rows after a long prefix and for the forms of q and out
that the kernel does not read or write in place. Host logic only: both routes
are replaced by recorders.
"""
import pytest

torch = pytest.importorskip("torch")

from tinytron_amd import ops
from tinytron_amd.cache import LayerPagedKVCache


@pytest.fixture
def route(monkeypatch):
    taken = []
    monkeypatch.setattr(ops, "prefill_attention_f32", lambda *a, **k: taken.append(("kernel", a, k)))
    monkeypatch.setattr(ops, "prefill_attention_rows", lambda *a, **k: taken.append(("rows", a, k)))

    def run(lens, new, Hq, Hkv, D, q=None, **kw):
        cache = LayerPagedKVCache(len(lens), Hkv, D, max(lens), 16, "cpu", torch.float32)
        cache.set_lengths(lens)
        cache.prefill_attend(torch.zeros(len(lens), Hq, max(new), D) if q is None else q, new, **kw)
        return taken.pop()

    return run


@pytest.mark.parametrize("lens,new,Hq,Hkv,D,expect", [
    ([6143], [6], 4, 1, 64, "kernel"),        # 24 rows, groups of 4: row attention from 6144 keys on
    ([6144], [6], 4, 1, 64, "rows"),
    ([6144], [7], 4, 1, 64, "kernel"),        # 28 rows
    ([6144], [8], 4, 1, 32, "rows"),          # 32 rows at head_dim 32
    ([6144], [9], 4, 1, 32, "kernel"),
    ([4095], [2], 4, 4, 64, "kernel"),        # one head a group: from 4096, past head_dim 64 from 2048
    ([4096], [2], 4, 4, 64, "rows"),
    ([2047], [2], 4, 4, 128, "kernel"),
    ([2048], [2], 4, 4, 128, "rows"),
    ([64, 6144], [0, 6], 4, 1, 64, "rows"),   # rows counted over the batch, keys by its longest sequence
    ([64, 6144], [1, 6], 4, 1, 64, "kernel"),
])
def test_few_rows_after_a_long_prefix(route, lens, new, Hq, Hkv, D, expect):
    assert route(lens, new, Hq, Hkv, D)[0] == expect


def test_forms_the_kernel_takes(route):
    lens, new, shape = [40, 23], [7, 4], (2, 4, 7, 32)
    args = (lens, new, 4, 2, 32)
    name, a, k = route(*args)
    assert name == "kernel" and a[2].tolist() == [33, 19] and k["new_lens"].tolist() == [7, 4] and a[3] == 40
    assert route(*args, q=torch.zeros(2, 7, 4, 32).transpose(1, 2))[0] == "kernel"
    assert route(*args, out=torch.zeros(2, 9, 4, 32)[:, 1:8])[0] == "kernel"
    for kw in (dict(q=torch.zeros(*shape, 2)[..., 0]), dict(out=torch.zeros(14, 4, 32)),
               dict(out=torch.zeros(2, 6, 4, 32)), dict(out=torch.zeros(2, 7, 4, 32, dtype=torch.bfloat16)),
               dict(out=torch.zeros(2, 7, 4, 32, 2)[..., 0]), dict(kernel=False)):
        name, a, k = route(*args, **kw)
        assert name == "rows" and a[2:4] == ([33, 19], [7, 4])
