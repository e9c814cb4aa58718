"""GPU parity: every workgroup shape that prefill attention picks, on both sides
of each line of its rule (keys within one tile or past it, columns for up to 4
waves or more, pairs up to what the GPU holds at once or past it: 256 CUs), for
ragged chunks over a page pool, unpadded and padded widths, 20 tokens past a
1024-token page-entry span. Reference: row attention, a kernel of its own.

Tolerance: the attention tests' bound against the exact result (2e-3 + 2e-2
|ref|) twice over, since both sides may be that far from it.
"""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DTYPE = {"bf16": torch.bfloat16, "fp8": torch.float8_e4m3fn}


def _cache(kind, B, Hkv, D, total, g):
    from tinytron_amd.cache import PagedLayerKVCache, random_page_table

    table, pages = random_page_table(total, 16, seed=B)
    c = PagedLayerKVCache(table, pages, Hkv, D, 16, "cuda", DTYPE[kind])
    for data, scale in ((c.layout.k, c.layout.k_scale), (c.layout.v, c.layout.v_scale)):
        if kind == "bf16":
            data.normal_(generator=g)
        else:  # every finite code, scales of up to 2 / 448
            codes = torch.randint(0, 254, data.shape, generator=g, device="cuda", dtype=torch.int16)
            data.copy_((codes + (codes >= 127)).to(torch.uint8))
            scale.copy_(torch.rand(scale.shape, generator=g, device="cuda") / 224)
    return c


@pytest.mark.parametrize("kind,D,G,Hkv,B,past,new", [
    # bf16, width 32: 8 x 64 to 512 pairs, 4 x 32 past them, 2 x 32 past 1024 with columns for two waves
    ("bf16", 32, 4, 8, 64, 70, 9), ("bf16", 32, 4, 8, 65, 70, 9), ("bf16", 24, 4, 8, 129, 70, 16),
    ("bf16", 32, 4, 8, 129, 70, 17), ("bf16", 32, 4, 8, 129, 70, 33), ("bf16", 32, 1, 16, 65, 3, 61),
    # width 64
    ("bf16", 64, 4, 8, 64, 70, 9), ("bf16", 64, 4, 8, 65, 70, 32), ("bf16", 40, 4, 8, 65, 70, 33),
    ("bf16", 64, 8, 2, 3, 4, 60), ("bf16", 48, 8, 2, 3, 5, 60),
    # width 128: 256 pairs
    ("bf16", 128, 4, 8, 32, 70, 9), ("bf16", 128, 4, 8, 33, 70, 32), ("bf16", 96, 3, 8, 33, 70, 41),
    ("bf16", 128, 16, 1, 2, 0, 64), ("bf16", 128, 16, 1, 2, 1, 64),
    # fp8, width 64: 768 pairs
    ("fp8", 64, 4, 16, 48, 70, 9), ("fp8", 64, 4, 16, 49, 70, 32), ("fp8", 48, 4, 16, 49, 70, 33),
    ("fp8", 64, 8, 2, 3, 4, 60),
    # fp8, width 128: a wave per pair for up to 64 keys or one wave's columns past 512 pairs; 4 x 64; 8 x 64
    ("fp8", 128, 4, 8, 2, 32, 32), ("fp8", 128, 4, 8, 2, 33, 32), ("fp8", 96, 6, 2, 3, 40, 20),
    ("fp8", 128, 4, 8, 65, 1200, 8), ("fp8", 96, 4, 8, 65, 500, 7), ("fp8", 128, 4, 8, 64, 70, 8),
    ("fp8", 128, 4, 8, 32, 70, 30), ("fp8", 128, 4, 8, 33, 70, 30), ("fp8", 80, 5, 4, 65, 70, 21),
    ("fp8", 128, 4, 2, 5, 1030, 150), ("fp8", 128, 4, 8, 17, 300, 100), ("fp8", 128, 4, 8, 17, 500, 100),
])
def test_shapes_against_row_attention(kind, D, G, Hkv, B, past, new):
    from tinytron_amd import ops

    g = torch.Generator(device="cuda").manual_seed(B + D + new)
    pick = torch.Generator().manual_seed(B)
    cached = [past] + torch.randint(0, past + 1, (B - 1,), generator=pick).tolist()
    news = [new] + torch.randint(0, new + 1, (B - 1,), generator=pick).tolist()
    c = _cache(kind, B, Hkv, D, [o + n for o, n in zip(cached, news)], g)
    q = torch.randn(B, Hkv * G, new, D, generator=g, device="cuda").bfloat16()
    out = torch.zeros(B, new, Hkv * G, D, device="cuda", dtype=torch.bfloat16)
    ops.prefill_attention(q, c.layout, torch.tensor(cached, dtype=torch.int32, device="cuda"), past + new,
                          new_lens=torch.tensor(news, dtype=torch.int32, device="cuda"), out=out)
    ref = ops.prefill_attention_rows(q, c.layout, cached, news).float()
    assert ((out.float() - ref).abs() <= 2 * (2e-3 + 2e-2 * ref.abs())).all()


def test_more_workgroups_than_one_launch_holds():
    # 2^24 + 5 sequences of one token (256 threads each: past 2^32), all on the one page of four cached tokens
    from tinytron_amd import ops

    B, D = 2 ** 24 + 5, 8
    g = torch.Generator(device="cuda").manual_seed(1)
    k, v = (torch.randn(16, D, generator=g, device="cuda").bfloat16() for _ in "kv")
    kv = ops.KVLayout(k=k.view(-1), v=v.view(-1), strides=(0, 16 * D, 16 * D), num_heads=1, head_dim=D, page_size=16,
                      capacity=16, kind="bf16", page_table=torch.zeros(B, 1, dtype=torch.int32, device="cuda"), num_pages=1)
    q = torch.randn(B, 1, 1, D, generator=g, device="cuda").bfloat16()
    got = ops.prefill_attention(q, kv, torch.full((B,), 3, dtype=torch.int32, device="cuda"), 4).view(B, D)
    for rows in (slice(0, 64), slice(2 ** 24 - 40, B)):
        scores = q.view(B, D)[rows].float() @ k[:4].float().t() / D ** 0.5
        ref = torch.softmax(scores, -1) @ v[:4].float()
        assert ((got[rows].float() - ref).abs() <= 2e-3 + 2e-2 * ref.abs()).all()


@pytest.mark.parametrize("D,B,past,new", [(128, 65, 100, 8), (128, 65, 1200, 3), (80, 130, 33, 4), (128, 3, 0, 20)])
def test_streaming_waves_repeat_themselves(D, B, past, new):
    # fp8 at width 128, a wave per pair with counted waits: lengths of odd and even numbers of 32-token tiles and of
    # 16-tile spans, each pass as the first one and as row attention
    from tinytron_amd import ops

    g = torch.Generator(device="cuda").manual_seed(D + B)
    pick = torch.Generator().manual_seed(past)
    cached = [past] + torch.randint(0, past + 1, (B - 1,), generator=pick).tolist()
    c = _cache("fp8", B, 8, D, [o + new for o in cached], g)
    q = torch.randn(B, 32, new, D, generator=g, device="cuda").bfloat16()
    pos = torch.tensor(cached, dtype=torch.int32, device="cuda")
    first = ops.prefill_attention(q, c.layout, pos, past + new)
    ref = ops.prefill_attention_rows(q, c.layout, cached, [new] * B).float()
    assert ((first.float() - ref).abs() <= 2 * (2e-3 + 2e-2 * ref.abs())).all()
    for _ in range(8):
        assert torch.equal(ops.prefill_attention(q, c.layout, pos, past + new), first)
