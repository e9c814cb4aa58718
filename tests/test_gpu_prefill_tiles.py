"""GPU parity: prefill attention at the edges of its workgroups: chunks ending
before, at and after a workgroup's 256 (128) (token, head) columns and a 64-key
tile, sequences ending inside one, keys past a 1024-token page-entry span, the
tile widths' padding, and the last and first batch of the two workgroup orders
(31, 32 and 40 (sequence, KV head) pairs). Tolerance as for the other prefill
attention tests (2e-3 + 2e-2 |ref|).
"""
import pytest

torch = pytest.importorskip("torch")

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


@pytest.mark.parametrize("G,D,fp8", [(4, 64, False), (1, 64, False), (16, 128, False), (3, 32, False),
                                     (4, 64, True), (8, 128, True)])
@pytest.mark.parametrize("past,token", [(0, 40), (0, 79), (21, 33), (50, 14)])
def test_infinite_value_stays_out_of_earlier_waves(G, D, fp8, past, token):
    # Value row `token` of a chunk of 80 is infinite (fp8: its codes NaN, its scale infinite). The tokens
    # of earlier waves (32 // G tokens each) share its 64-key tile and must not see it, bit for bit.
    from tinytron_amd import ops

    g = torch.Generator(device="cuda").manual_seed(D + G)
    Hkv, new, cap = 2, 80, 144
    rows = Hkv * cap
    q = torch.randn(1, Hkv * G, new, D, generator=g, device="cuda").bfloat16()
    kw = {}
    if fp8:
        k, v = (torch.randn(rows, D, generator=g, device="cuda").to(torch.float8_e4m3fn).view(torch.uint8) for _ in "kv")
        scale = torch.rand(2 * rows, generator=g, device="cuda") + 0.5  # groups of 16 K scales, then 16 V scales
        kw = dict(k_scale=scale, v_scale=scale[16:])
    else:
        k, v = (torch.randn(rows, D, generator=g, device="cuda").bfloat16() for _ in "kv")

    def run():
        kv = ops.KVLayout(k=k.view(-1), v=v.view(-1), strides=(Hkv * cap * D, 16 * D, cap * D), num_heads=Hkv,
                          head_dim=D, page_size=16, capacity=cap, kind="fp8" if fp8 else "bf16", **kw)
        return ops.prefill_attention(q, kv, torch.tensor([past], dtype=torch.int32, device="cuda"), past + new)

    plain = run()
    for h in range(Hkv):
        r = h * cap + past + token
        if fp8:
            v[r] = 0x7F
            scale[r + r // 16 * 16 + 16] = float("inf")
        else:
            v[r] = float("inf")
    got = run()
    first = token // (32 // G) * (32 // G)  # of the token's wave
    assert torch.isfinite(plain.float()).all()
    assert torch.equal(got[:, :first], plain[:, :first])
    assert not torch.isfinite(got[:, token:].float()).any()
