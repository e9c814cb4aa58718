"""GPU parity of the decode-step layer kernels' row tiles: 16-, 32- and 64-row
tiles of the split-K and SwiGLU GEMMs at their edges (the same row must come
out bit for bit from every tile: the contraction order does not change), the
1280-wide chunks, and the 1024-thread residual add + RMSNorm (rows wider than
2048 with more than four splits).

Tolerances: GEMM partials 1e-5 (|x| . |W|^T) of fp64 (fp32 sums of at most 1280
products); RMSNorm one bf16 ulp of the fp64 result, the residual bit for bit
(the splits are added in order).
"""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf16(g, *shape, scale=1.0):
    return (torch.randn(shape, generator=g) * scale).to(torch.bfloat16)


@pytest.mark.parametrize("N,K,kc", [(192, 512, 256), (128, 1024, 512), (64, 2048, 1024), (192, 2560, 1280)])
@pytest.mark.parametrize("packed", [False, True])
def test_row_tiles_of_the_split_gemm(N, K, kc, packed):
    from tinytron_amd import ops

    g = torch.Generator().manual_seed(N + K)
    x, w = _bf16(g, 33, K), _bf16(g, N, K)
    wd = ops.PackedWeight(w.to(DEV)) if packed else w.to(DEV)
    sizes = [1, 15, 16, 17, 32] + ([33] if kc <= 1024 else [])
    outs = {m: ops.linear_partials(x[:m].to(DEV), wd, k_chunk=kc).cpu() for m in sizes}
    full = outs[sizes[-1]]
    for m, p in outs.items():
        assert p.shape == (K // kc, m, N) and torch.equal(p, full[:, :m])
    xc = x[:sizes[-1]].double().view(-1, K // kc, kc)
    wc = w.double().view(N, K // kc, kc)
    for s in range(K // kc):
        ref = xc[:, s] @ wc[:, s].t()
        bound = 1e-5 * (xc[:, s].abs() @ wc[:, s].abs().t())
        assert ((full[s].double() - ref).abs() <= bound).all()


def test_wide_chunks_need_few_rows():
    from tinytron_amd import ops

    g = torch.Generator().manual_seed(1)
    with pytest.raises(ValueError, match="k_chunk"):
        ops.linear_partials(_bf16(g, 33, 1280).to(DEV), _bf16(g, 64, 1280).to(DEV), k_chunk=1280)


@pytest.mark.parametrize("K,inter", [(768, 48), (1024, 32), (2048, 24), (2048, 64)])
def test_row_tiles_of_the_swiglu_gemm(K, inter):
    from tinytron_amd import ops

    g = torch.Generator().manual_seed(K + inter)
    x, wg, wu = _bf16(g, 65, K), _bf16(g, inter, K, scale=0.05), _bf16(g, inter, K, scale=0.05)
    w = ops.PackedWeight(ops.interleave_gate_up(wg, wu).to(DEV))
    outs = {m: ops.linear_swiglu(x[:m].to(DEV), w).cpu() for m in (1, 16, 17, 32, 33, 64, 65)}
    for m, a in outs.items():
        assert torch.equal(a, outs[65][:m]), m
    gate, up = x.double() @ wg.double().t(), x.double() @ wu.double().t()
    gate, up = gate.to(torch.bfloat16).double(), up.to(torch.bfloat16).double()
    ref = torch.nn.functional.silu(gate).to(torch.bfloat16).double() * up
    # three bf16 roundings of values that can each fall one ulp apart: 3 x 2^-8, and of gate near 0
    err = (outs[65].double() - ref).abs()
    assert (err <= 3 * 2.0 ** -8 * ref.abs() + 2.0 ** -7 * up.abs() * 0.05).all()


@pytest.mark.parametrize("C,S", [(2052, 5), (4096, 16), (4096, 17), (5120, 8), (5120, 27), (8192, 9), (8188, 33)])
@pytest.mark.parametrize("M", [1, 3])
def test_wide_residual_norm(C, S, M):
    from tinytron_amd import ops

    g = torch.Generator().manual_seed(C + S)
    x, w = torch.randn(M, C, generator=g), torch.randn(C, generator=g)
    P = torch.randn(S, M, C, generator=g)
    xd = x.to(DEV)
    y = ops.add_rmsnorm(xd, w.to(DEV), 1e-6, partials=P.to(DEV)).cpu().double()
    acc = P[0].clone()
    for s in range(1, S):
        acc += P[s]
    res = x + acc.to(torch.bfloat16).float()
    assert torch.equal(xd.cpu(), res)
    ref = w.double() * res.double() * torch.rsqrt(res.double().square().mean(-1, keepdim=True) + 1e-6)
    assert ((y - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-6).all()
