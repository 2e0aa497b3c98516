"""The 192 x 192-tile products (csrc/tile192.hip): the chunked weight
gradients at the edges of their chunks, tiles and experts, against fp64.

Bound per element: one bf16 rounding of the result (2^-9 relative, 2^-8 taken)
plus the fp32 accumulation of n products, n * 2^-24 of the sum of their
magnitudes, whatever the order.
"""
import pytest
import torch

from uttt_amd.lact_moe_triton import _grouped as G

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (group sizes per batch, D, I, N or None): chunks start at 512 tokens (at
# least 2 D) for D, I <= 512; wider experts take them with short segments
WGRAD = {
    "chunk_edges": ([[512, 513, 0, 511, 1024, 1025, 31, 1]], 192, 192, None),
    "ragged_widths_two_batches": ([[700, 0, 1300], [1, 1999, 0]], 200, 104, None),
    "over_64_experts": ([[17 * (i % 5) for i in range(70)]], 64, 8, None),
    "slack_rows": ([[600, 40, 900]], 384, 384, 1700),
    "over_count": ([[600, 900, 700]], 96, 200, 1400),      # clamped to N tokens
    "wide_short": ([[3, 200, 0, 129, 64, 33, 1, 250]], 520, 776, None),
    "all_empty": ([[0, 0, 0]], 192, 384, 64),
    "long": ([[9000, 2, 5000]], 64, 128, None),
}


@pytest.mark.parametrize("name", list(WGRAD))
def test_chunked_weight_gradients(name):
    sizes, D, I, N = WGRAD[name]
    gs = torch.tensor(sizes, dtype=torch.int32)
    B, E = gs.shape
    N = int(gs.sum(1).max()) if N is None else N
    g = torch.Generator().manual_seed(N)
    dy, k, hid, v = (torch.randn(B, N, w, generator=g).to(torch.bfloat16).to(DEV)
                     for w in (2 * I, D, I, D))
    dw02, dw1 = G.wgrad_pair(dy, k, hid, v, gs.to(DEV))
    again = G.wgrad_pair(dy, k, hid, v, gs.to(DEV))
    assert torch.equal(dw02, again[0]) and torch.equal(dw1, again[1])
    for b in range(B):
        start = 0
        for e in range(E):
            n = max(0, min(int(gs[b, e]), N - start))
            s = slice(start, start + n)
            start += n
            for ours, p, q in ((dw02[b, e], dy, k), (dw1[b, e], v, hid)):
                p64, q64 = p[b, s].double(), q[b, s].double()
                ref = p64.T @ q64
                bound = 2.0 ** -8 * ref.abs() + n * 2.0 ** -24 * (p64.abs().T @ q64.abs())
                assert bool(((ours.double() - ref).abs() <= bound).all()), (b, e, n)
