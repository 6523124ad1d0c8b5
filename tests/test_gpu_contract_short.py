"""GPU: the mixed contraction at short K on shapes that two 64 x 128 tiles per CU cover: the k-interleaved
operands through the direct-load kernel, the same bits as the plain layout, at ragged edges and on both
sides of the K at which the staged tiles take over."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P,n,K64,K32", [(16384, 200, 64, 336), (16100, 193, 5, 16), (16383, 255, 0, 512),
                                         (16384, 200, 3, 528), (8190, 400, 1, 272), (15300, 256, 2, 48)])
def test_short_k_same_bits_as_the_plain_layout(gpu, P, n, K64, K32):
    from smolyax_amd import _native as N

    g = torch.Generator(device="cuda").manual_seed(P + n + K32)
    A64 = torch.randn((max(K64, 1), P), dtype=torch.float64, device="cuda", generator=g)
    B64 = torch.randn((max(K64, 1), n), dtype=torch.float64, device="cuda", generator=g)
    A32 = torch.randn((K32, P), dtype=torch.float32, device="cuda", generator=g)
    B32 = torch.randn((K32, n), dtype=torch.float32, device="cuda", generator=g)
    off = torch.randn(n, dtype=torch.float64, device="cuda", generator=g)
    k4 = lambda M: M.view(K32 // 4, 4, M.shape[1]).permute(0, 2, 1).contiguous()
    A4, B4 = k4(A32), k4(B32)
    st = torch.cuda.current_stream().cuda_stream
    out = []
    for name, a, b in (("sbi_contract_split", A32, B32), ("sbi_contract_split_k4", A4, B4)):
        Y = torch.full((P, n), float("nan"), dtype=torch.float64, device="cuda")
        N.check(N.fn[name](A64.data_ptr(), P, B64.data_ptr(), n, K64, a.data_ptr(), P, b.data_ptr(), n,
                           K32, off.data_ptr(), Y.data_ptr(), n, P, n, st), name)
        out.append(Y)
    assert torch.equal(out[0], out[1])
