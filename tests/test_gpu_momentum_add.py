"""The momentum sum g + mom * m_coeff[b] on both kernels: whole aligned vectors
and the scalar one.  Bit-exact: one product and one sum, each rounded to fp32."""
import pytest
import torch

from uttt_amd import fast_weight_write as fww

pytestmark = pytest.mark.gpu


# one vector, around half a workgroup tile of 4096 (below it the scalar kernel), a
# whole tile, one vector past it,
# several tiles, and counts that are no whole vectors
@pytest.mark.parametrize("n", [4, 2044, 2048, 2052, 4096, 4100, 3 * 4096 + 12, 1, 4099])
@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("offset", [0, 1])
def test_momentum_sum(n, B, dtype, offset):
    gen = torch.Generator().manual_seed(n + B)
    g = torch.randn(B * n, generator=gen).to(dtype)
    mom, c = torch.randn(B * n, generator=gen), torch.randn(B, generator=gen)

    def place(t):  # `offset` elements past an aligned start
        buf = torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda")[offset:]
        return buf.copy_(t).view(B, 1, 1, n)

    out = fww._momentum(place(g), place(mom), c.cuda())
    ref = g.view(B, n).float() + mom.view(B, n) * c[:, None]
    assert torch.equal(out.cpu().view(B, n), ref)
