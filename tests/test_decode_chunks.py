"""Split-K chunk widths of a decode step's projections. Host logic only."""
from types import SimpleNamespace

import pytest

torch = pytest.importorskip("torch")

from tinytron_amd import model


def _chunks(monkeypatch, cus, C, inter, B):
    monkeypatch.setattr(model, "_cu_count", lambda device: cus)
    gpt = SimpleNamespace(config=SimpleNamespace(hidden_size=C, intermediate_size=inter), _k_chunk=model.GPT._k_chunk,
                          wte=SimpleNamespace(weight=torch.empty(0)))
    return model.GPT._chunks(gpt, B)


@pytest.mark.parametrize("cus,C,inter,B,expect", [
    (256, 2048, 6144, 64, (512, 256, 1024, 512)),    # gate|up: 128 x 2 workgroups of 96 rows
    (256, 2048, 6912, 64, (512, 256, 512, 256)),     # 144 x 2
    (256, 5120, 13824, 5, (1280, 512, 1024, 512)),
    (256, 5120, 13824, 64, (512, 512, 512, 512)),
    (128, 2048, 6144, 64, (512, 256, 512, 512)),     # half the CUs do not take gate|up whole,
    (32, 2048, 6144, 64, (512, 512, 512, 512)),      # an eighth has c_proj's workgroups at 512
    (256, 1024, 8192, 64, (512, 256, 1024, 512)),    # N 16384: no 96-row workgroups; 128 of 128
    (128, 1024, 8192, 64, (512, 256, 1024, 512)),    # 128 of 128 on 128 CUs
    (127, 1024, 8192, 64, (512, 256, 512, 512)),
])
def test_chunks_follow_the_device(monkeypatch, cus, C, inter, B, expect):
    assert _chunks(monkeypatch, cus, C, inter, B) == expect
