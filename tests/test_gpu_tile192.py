"""The 192 x 192-tile products (csrc/tile192.hip): the chunked weight
gradients at the edges of their chunks, tiles and experts, against fp64, and
the Newton-Schulz steps.

Bound of the gradients per element: one bf16 rounding of the result (2^-9 relative, 2^-8 taken)
plus the fp32 accumulation of n products, n * 2^-24 of the sum of their
magnitudes, whatever the order.
"""
import pytest
import torch

from oracle import write as OW
from uttt_amd import _lib as L
from uttt_amd import fast_weight_write as FWW
from uttt_amd.lact_moe_triton import _grouped as G

pytestmark = pytest.mark.gpu
DEV = "cuda"

# (group sizes per batch, D, I, N or None): pieces start at 512 tokens (at
# least 2 D) for D, I <= 512, else at 4096; some sizes take whole segments on
# the 256 x 256 tiles (wg192_plan)
WGRAD = {
    "chunk_edges": ([[512, 513, 0, 511, 1024, 1025, 31, 1]], 192, 192, None),
    "ragged_widths_two_batches": ([[700, 0, 1300], [1, 1999, 0]], 200, 104, None),
    "over_64_experts": ([[17 * (i % 5) for i in range(70)]], 64, 8, None),
    "slack_rows": ([[600, 40, 900]], 384, 384, 1700),
    "over_count": ([[600, 900, 700]], 96, 200, 1400),      # clamped to N tokens
    "wide_short": ([[3, 200, 0, 129, 64, 33, 1, 250]], 520, 776, None),
    "all_empty": ([[0, 0, 0]], 192, 384, 64),
    "long": ([[9000, 2, 5000]], 64, 128, None),
    "pieces_ragged_widths": ([[700, 0, 1300] + [0] * 5, [1, 1999, 0] + [0] * 5], 200, 104, None),
    "pieces_slack_rows": ([[600, 40, 900, 0, 0]], 384, 384, 1700),
    "pieces_over_count": ([[600, 900, 700, 0, 0, 0]], 96, 200, 1400),
    "pieces_long": ([[9000, 2, 5000] + [0] * 53], 64, 128, None),
    "pieces_deep": ([[8300, 0, 60] + [1] * 30], 2056, 8, None),   # pieces of 2 D or more tokens
    "few_chunks": ([[0, 250]], 1544, 264, None),   # tiles of one dealt to the XCDs
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


@pytest.mark.parametrize("name", list(WGRAD))
def test_weight_gradients_equal_general_tiles(name):
    """The forced 256 x 256 tiles (whole segments, or split K over few tiles):
    the same products, an expert of several pieces added in another order."""
    sizes, D, I, N = WGRAD[name]
    gs = torch.tensor(sizes, dtype=torch.int32, device=DEV)
    B, E = gs.shape
    N = int(gs.sum(1).max()) if N is None else N
    g = torch.Generator().manual_seed(N)
    ins = [torch.randn(B, N, w, generator=g).to(torch.bfloat16).to(DEV) for w in (2 * I, D, I, D)]
    ours = G.wgrad_pair(*ins, gs)
    prev = L.lib().uttt_debug_set_gemm_layout(2)
    try:
        whole = L.lib().uttt_grouped_wgrad_pair_workspace_bytes(B, E, I, D, N) == 0
        general = G.wgrad_pair(*ins, gs)
    finally:
        L.lib().uttt_debug_set_gemm_layout(prev)
    for a, b in zip(ours, general):
        for e in range(E):
            n = int(gs[:, e].max())
            x, y = a[:, e].double(), b[:, e].double()
            if whole and n <= 512:   # one piece on either side: the same chain of products
                assert torch.equal(x, y), e
            else:                    # as above: one rounding each, sums in two orders
                assert bool(((x - y).abs() <= 2.0 ** -7 * y.abs() + n * n * 2.0 ** -23).all()), e


def test_weight_gradients_of_many_batches():
    """More than 65 535 (batch, expert) pairs, segments of two pieces among them."""
    B, E, D, I, N = 1024, 65, 8, 8, 520
    g = torch.Generator().manual_seed(2)
    gs = torch.zeros(B, E, dtype=torch.int32)
    gs[:, 0], gs[:, 64] = 3, 517          # the last expert's segment starts at 3
    dy, k, hid, v = (torch.randint(-2, 3, (B, N, w), generator=g).to(torch.bfloat16).to(DEV)
                     for w in (2 * I, D, I, D))
    dw02, dw1 = G.wgrad_pair(dy, k, hid, v, gs.to(DEV))
    for e, s in ((0, slice(0, 3)), (64, slice(3, 520))):   # small whole numbers: exact sums
        for ours, p, q in ((dw02, dy, k), (dw1, v, hid)):
            pt = p[:, s].float().transpose(1, 2).contiguous()
            ref = torch.bmm(pt, q[:, s].float().contiguous())
            assert torch.equal(ours[:, e].float(), ref.to(torch.bfloat16).float())
    assert torch.count_nonzero(dw02[:, 1:64]) == 0 and torch.count_nonzero(dw1[:, 1:64]) == 0


@pytest.mark.parametrize("given", ["none", "short", "unaligned"])
def test_weight_gradients_without_room_for_partials(given):
    """48 experts of 192 x 192 with segments of several chunks: the workspace is
    optional, and without it every segment is summed whole."""
    B, E, D, I, N = 1, 48, 192, 192, 48 * 700
    g = torch.Generator().manual_seed(1)
    sizes = torch.randint(0, 1400, (B, E), generator=g, dtype=torch.int32)
    gs = sizes.to(DEV)
    dy, k, hid, v = (torch.randn(B, N, w, generator=g).to(torch.bfloat16).to(DEV)
                     for w in (2 * I, D, I, D))
    need = L.lib().uttt_grouped_wgrad_pair_workspace_bytes(B, E, I, D, N)
    assert need > 0
    ws = torch.empty(need + 16, dtype=torch.uint8, device=DEV)
    ptr, size = {"none": (None, 0), "short": (L.ptr(ws), need - 1),
                 "unaligned": (L.ptr(ws) + 4, need)}[given]
    dw02 = torch.empty(B, E, 2 * I, D, dtype=torch.bfloat16, device=DEV)
    dw1 = torch.empty(B, E, D, I, dtype=torch.bfloat16, device=DEV)
    L.call("uttt_grouped_wgrad_pair", L.ptr(dy), L.ptr(k), L.ptr(hid), L.ptr(v), L.ptr(gs), B, E,
           I, D, N, L.ptr(dw02), L.ptr(dw1), ptr, size, L.stream_of(k))
    ref = G.wgrad_pair(dy, k, hid, v, gs)
    # one bf16 rounding each, and the fp32 sums in two orders of n products of
    # mean magnitude 2 / pi: twice n 2^-24 times n of them
    n = int(sizes.max())
    for a, b in zip((dw02, dw1), ref):
        a, b = a.double(), b.double()
        assert bool(((a - b).abs() <= 2.0 ** -7 * b.abs() + n * n * 2.0 ** -23).all())


# (matrices, rows, columns, dtype, offset in elements): partial tiles on both
# axes, more matrices than XCDs, several tiles per side (mirrored ones), a side
# below one MFMA block, an input that is not 16-byte aligned
@pytest.mark.parametrize("n,R,C,dtype,offset", [
    (5, 200, 264, torch.float32, 0), (9, 384, 384, torch.bfloat16, 0),
    (2, 776, 392, torch.float32, 0), (3, 8, 1000, torch.bfloat16, 0),
    (1, 584, 584, torch.float32, 0), (2, 208, 416, torch.float32, 1),
    (2, 416, 208, torch.bfloat16, 1),
    (1, 1544, 1608, torch.float32, 0),   # a second band of tiles, one matrix on every XCD
])
def test_newton_schulz5_tiles(n, R, C, dtype, offset):
    """Against the same iteration in fp64: overall no further off than 1.5x the
    bf16 oracle (both are bf16 realisations of one map), and at most 5e-2 of
    the rms row (column) norm in every row and column of 200 elements or more.
    A perturbation grows by up to a = 4 per step along
    a small singular direction, so two realisations differ by about 1e-2,
    spread evenly over the rows, and no elementwise bound of a few ulps holds;
    an element that is wrong by its own size is 1 / sqrt(side) of its row, at
    least 5e-2 for the sides up to 392."""
    G = torch.randn(n, R, C, generator=torch.Generator().manual_seed(R + C)).to(dtype)
    buf = torch.empty(n * R * C + offset, dtype=dtype, device=DEV)
    dev = buf[offset:].view(n, R, C)
    dev.copy_(G)
    ours = FWW.newton_schulz5(dev, 0.75).cpu().double()
    ref = (OW.newton_schulz5(G) * 0.75).double()
    X = G.double()
    X = X.transpose(1, 2) if R > C else X
    X = X / (X.norm(dim=(1, 2), keepdim=True) + 1e-7)
    for a, b, c in OW.NS5_COEFFS:
        A = X @ X.transpose(1, 2)
        X = a * X + (b * A + c * A @ A) @ X
    exact = (X.transpose(1, 2) if R > C else X) * 0.75
    rel = lambda x: ((x - exact).norm() / exact.norm()).item()
    assert rel(ours) <= 1.5 * rel(ref) + 1e-3
    for dim in (1, 2):
        if exact.shape[dim] >= 200:
            rms = exact.norm(dim=dim).pow(2).mean().sqrt()
            assert ((ours - exact).norm(dim=dim).max() / rms).item() <= 5e-2


@pytest.mark.parametrize("n,R,C", [(9, 392, 584), (3, 1544, 1608)])
def test_newton_schulz5_alone_or_stacked(n, R, C):
    """A matrix's result does not depend on the matrices beside it: the tiles of
    all are cut into one run per XCD, of which one alone fills parts (several
    tiles per side; past eight a second band)."""
    G = torch.randn(n, R, C, generator=torch.Generator().manual_seed(n)).to(DEV)
    all_ = FWW.newton_schulz5(G)
    for i in range(n):
        assert torch.equal(FWW.newton_schulz5(G[i:i + 1].contiguous())[0], all_[i])
